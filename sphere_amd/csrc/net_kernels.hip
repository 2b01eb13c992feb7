// net_kernels.hip -- gfx950 kernels of the Darcy correction network: 3x3x3
// convolutions (stride 1, zero padding 1) as implicit GEMMs on the matrix
// cores (v_mfma_f32_16x16x32_bf16 for the forward pass, 16x16x16 for the
// weight gradients: BF16 operands, FP32 accumulation), their
// data and weight gradients, 2x average pooling, nearest upsampling with a
// skip add, and the ReLU mask.
//
// Activations are channels-last, act[v * C + c] with v = (z * ny + y) * nx
// + x, BF16 bit patterns (uint16_t) for the matrix-core operands and FP32
// for gradients that are summed from several paths.  Weights are
// w[tap][co][ci], tap = (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1), so that four
// consecutive input channels of one tap and output channel are one 8-byte
// load.
#include "net_kernels.h"

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// gfx950's v_mfma_f32_16x16x32_bf16: A[m][k] with m = lane % 16 and k = 8
// (lane / 16) + 0..7 (eight BF16 per lane), B[k][n] with n = lane % 16 and k
// likewise, D as for the 16x16x16 shape.  Half the instructions, and half
// the dependent steps of a K loop, of the 16x16x16 shape.
__device__ __forceinline__ f32x4 mfma32(s16x8 a, s16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ s16x8 cat8(bf16x4 lo, bf16x4 hi)
{
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}


// neighbour (x, y, z) of the 3x3x3 stencil: wrapped along periodic axes,
// false where it falls in the zero padding
__device__ __forceinline__ bool nb_in(const NetGeom &g, int &x, int &y, int z)
{
    const int nx = (int)g.nx, ny = (int)g.ny;
    if (g.wrap & 1u) x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
    if (g.wrap & 2u) y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
    return x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < (int)g.nz;
}

__device__ __forceinline__ void vox_xyz(const NetGeom &g, uint32_t v, int &x, int &y, int &z)
{
    x = (int)(v % g.nx);
    const uint32_t r = v / g.nx;
    y = (int)(r % g.ny);
    z = (int)(r / g.ny);
}

// ---------------------------------------------------------------------------
// Forward convolution.  A wave computes MT 16-voxel M tiles by all 16*NT
// output channels; K runs over 32-wide steps: two (tap, 16-channel chunk)
// pairs of the input (CIN4: inputs of 4 channels, eight taps per step, two
// per 16-lane group).  With KS > 1 the KS waves of a block share the M
// tiles and take every KS-th step, and their partial sums meet in LDS
// (small grids: more waves, shorter chains).  Each wave issues the loads of
// G steps before their MFMAs.  MFMA 16x16x32 lane layout: A[m][k] with
// m = lane % 16, k = 8 (lane / 16) + 0..7; B[k][n] with n = lane % 16, k
// likewise; the accumulator holds D[4 (lane / 16) + i][lane % 16].
// ---------------------------------------------------------------------------
#define CONV_G 4
// K split of the grids of at most CONV_SMALL_V voxels: CONV_KS_SMALL waves
// per 16-voxel tile (4 on larger grids below 65536 voxels).  On the network's
// 48 x 48 x 96 grid, 8 waves on its two coarsest levels took one forward pass
// from 154 to 144 us; 16 waves, or 8 on the 27,648-voxel level too, were
// slower, except for inputs of 64 channels (143.4 us).
#define CONV_SMALL_V 8192u
#define CONV_KS_SMALL 8

// Epilogue of the convolutions: acc[j][t] holds, for M tile j (16
// voxels from vbase[j] along x), voxels vbase[j] + 4 grp + i (i = 0..3) and
// output channel 16 t + m.
// The children of coarse voxel v on the grid twice as fine, channel co:
// yfine = a + skip, for children k0, k0 + dk, ... (k < 8)
__device__ __forceinline__ void up_children(const NetGeom &g, uint32_t v, int co, int cout_real, float av,
                                            int k0, int dk, const uint16_t *__restrict__ skip,
                                            uint16_t *__restrict__ yfine)
{
    int x, y, z;
    vox_xyz(g, v, x, y, z);
    const uint32_t fnx = 2u * g.nx, fny = 2u * g.ny;
    for (int k = k0; k < 8; k += dk) {
        const uint32_t fv = ((2u * z + (k >> 2)) * fny + 2u * y + ((k >> 1) & 1)) * fnx + 2u * x + (k & 1);
        const size_t fo = (size_t)fv * cout_real + co;
        yfine[fo] = f2bf(av + bf2f(skip[fo]));
    }
}

template <int NT, int MT>
__device__ __forceinline__ void conv_store(const f32x4 (&acc)[MT][NT], const uint32_t (&vbase)[MT], uint32_t V,
                                           uint32_t m, uint32_t grp, const float *__restrict__ bias,
                                           int cout_real, void *__restrict__ out, int mode,
                                           const float *__restrict__ proj, float *__restrict__ out2,
                                           const NetGeom &g, const uint16_t *__restrict__ skip,
                                           uint16_t *__restrict__ yfine)
{
    if (NT == 1 && mode == NET_OUT_PROJ) {
        // h = bf16(relu(acc + bias)) stored, and out2[v] = sum_c h[v][c]
        // proj[c] + proj[16]: the 16 channels of a voxel sit in the 16 lanes
        // of one lane group, summed by xor shuffles within the group
        const float bv = bias[m];
        const float wp = proj[m];
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t v = vbase[j] + 4u * grp + (uint32_t)i;
                const float r = acc[j][0][i] + bv;
                const uint16_t h = f2bf(r > 0.f ? r : 0.f);
                float sum = bf2f(h) * wp;
                sum += __shfl_xor(sum, 1);
                sum += __shfl_xor(sum, 2);
                sum += __shfl_xor(sum, 4);
                sum += __shfl_xor(sum, 8);
                if (v < V) {
                    ((uint16_t *)out)[(size_t)v * 16 + m] = h;
                    if (m == 0) out2[v] = sum + proj[16];
                }
            }
        return;
    }
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int co = t * 16 + (int)m;
            if (co >= cout_real) continue;
            const float bv = bias ? bias[co] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t v = vbase[j] + 4u * grp + (uint32_t)i;
                if (v >= V) continue;
                float r = acc[j][t][i] + bv;
                const size_t o = (size_t)v * cout_real + co;
                if (mode == NET_OUT_BF16_RELU || mode == NET_OUT_RELU_UP) {
                    const uint16_t a = f2bf(r > 0.f ? r : 0.f);
                    ((uint16_t *)out)[o] = a;
                    if (mode == NET_OUT_RELU_UP && yfine)  // the 8 children: a + skip
                        up_children(g, v, co, cout_real, bf2f(a), 0, 1, skip, yfine);
                } else if (mode == NET_OUT_F32) {
                    ((float *)out)[o] = r;
                } else {
                    ((float *)out)[o] += r;
                }
            }
        }
}


template <int NT, int MT, int KS, bool CIN4>
__device__ __forceinline__ void conv_fwd_body(const NetGeom &g, const uint16_t *__restrict__ in, int cin,
                                              const uint16_t *__restrict__ w,
                                              const float *__restrict__ bias, int cout_real,
                                              void *__restrict__ out, int mode,
                                              const float *__restrict__ proj, float *__restrict__ out2,
                                              const uint16_t *__restrict__ skip,
                                              uint16_t *__restrict__ yfine, uint32_t bid, uint32_t nblk)
{
    __shared__ float red[KS > 1 ? (KS - 1) * MT * NT * 4 * 64 : 1];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    // each XCD works through one contiguous range of tiles, whose stencil
    // reads then mostly hit that XCD's L2
    const uint32_t b = xcd_tile(bid, nblk);
    const uint32_t tile = KS == 1 ? b * 4u + wv : b;
    const int kpart = KS == 1 ? 0 : (int)wv;
    const uint32_t V = g.nx * g.ny * g.nz;
    const uint32_t v0 = tile * 16u * MT;
    if (v0 >= V) return;  // uniform over the block when KS > 1
    const uint32_t m = lane & 15u, grp = lane >> 4;
    const int cout = 16 * NT;
    const int nx = (int)g.nx, ny = (int)g.ny;
    int vx[MT], vy[MT], vz[MT];
    bool vin[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const uint32_t v = v0 + 16u * j + m;
        vin[j] = v < V;
        vox_xyz(g, vin[j] ? v : 0u, vx[j], vy[j], vz[j]);
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // K runs over 32-wide steps u.  Inputs of 16k channels: 16-channel steps
    // st = (tap, chunk) taken in pairs, lane group grp reading channels
    // 8 (grp & 1) .. + 7 of step 2u + (grp >> 1).  Inputs of 4 channels: taps
    // 8u + 2 grp and 8u + 2 grp + 1, four channels each.
    const int chunks = CIN4 ? 1 : (cin >> 4);
    const int S = CIN4 ? 27 : 27 * chunks;
    const int U = CIN4 ? 4 : (S + 1) / 2;
    const int half = (int)(grp & 1u), sub = (int)(grp >> 1);
    const int cs = CIN4 ? 4 : cin;
    const s16x8 zero8 = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    for (int u0 = kpart; u0 < U; u0 += KS * CONV_G) {
        s16x8 a[CONV_G][MT], b[CONV_G][NT];
#pragma unroll
        for (int q = 0; q < CONV_G; ++q) {
            const int u = u0 + q * KS;
            if (CIN4) {
                bf16x4 bl[NT][2], al[MT][2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int tap = 8 * u + 2 * (int)grp + e;
                    const bool tok = u < U && tap < 27;
                    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        bl[t][e] = bf16x4{0, 0, 0, 0};
                        if (tok) bl[t][e] = *(const bf16x4 *)(w + ((size_t)(tap * cout + t * 16 + (int)m) * 4));
                    }
#pragma unroll
                    for (int j = 0; j < MT; ++j) {
                        int x = vx[j] + dx, y = vy[j] + dy;
                        const int z = vz[j] + dz;
                        al[j][e] = bf16x4{0, 0, 0, 0};
                        if (tok && vin[j] && nb_in(g, x, y, z))
                            al[j][e] = *(const bf16x4 *)(in + ((size_t)((z * ny + y) * nx + x) * 4));
                    }
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) b[q][t] = cat8(bl[t][0], bl[t][1]);
#pragma unroll
                for (int j = 0; j < MT; ++j) a[q][j] = cat8(al[j][0], al[j][1]);
            } else {
                const int st = 2 * u + sub;
                const bool tok = u < U && st < S;
                const int tap = st / chunks;
                const int ci = (st - tap * chunks) * 16 + 8 * half;
                const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    b[q][t] = zero8;
                    if (tok) b[q][t] = *(const s16x8 *)(w + ((size_t)(tap * cout + t * 16 + (int)m) * cs + ci));
                }
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    int x = vx[j] + dx, y = vy[j] + dy;
                    const int z = vz[j] + dz;
                    a[q][j] = zero8;
                    if (tok && vin[j] && nb_in(g, x, y, z))
                        a[q][j] = *(const s16x8 *)(in + ((size_t)((z * ny + y) * nx + x) * cs + ci));
                }
            }
        }
#pragma unroll
        for (int q = 0; q < CONV_G; ++q) {
            if (u0 + q * KS >= U) break;
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[j][t] = mfma32(a[q][j], b[q][t], acc[j][t]);
        }
    }
    if (KS > 1) {
        if (wv > 0) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        red[((((wv - 1) * MT + j) * NT + t) * 4 + i) * 64 + lane] = acc[j][t][i];
        }
        __syncthreads();
        if (mode != NET_OUT_RELU_UP && wv > 0) return;
        if (wv == 0) {
#pragma unroll 1
            for (int k = 0; k < KS - 1; ++k)
#pragma unroll
                for (int j = 0; j < MT; ++j)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[j][t][i] += red[(((k * MT + j) * NT + t) * 4 + i) * 64 + lane];
        }
        if (mode == NET_OUT_RELU_UP) {
            // wave 0 stores the coarse output and puts a = bf16(relu(acc +
            // bias)) in LDS, from which all waves write the 8 children
            __shared__ float s_a[MT * NT * 4][64];
            uint32_t vb[MT];
#pragma unroll
            for (int j = 0; j < MT; ++j) vb[j] = v0 + 16u * j;
            if (wv == 0) {
                conv_store<NT, MT>(acc, vb, V, m, grp, bias, cout_real, out, NET_OUT_RELU_UP, proj, out2, g,
                                   skip, nullptr);
#pragma unroll
                for (int j = 0; j < MT; ++j)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const int co = t * 16 + (int)m;
                        const float bv = (bias && co < cout_real) ? bias[co] : 0.f;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float r = acc[j][t][i] + bv;
                            s_a[(j * NT + t) * 4 + i][lane] = bf2f(f2bf(r > 0.f ? r : 0.f));
                        }
                    }
            }
            __syncthreads();
            // then each lane writes 8 channels (16 B) of one child: item =
            // ((voxel * 8 + child) * cout_real / 8 + channel octet), so
            // neighbouring lanes fill whole fine-voxel rows (cout_real % 8 == 0)
            const int octets = cout_real >> 3;
            const int items = 16 * MT * 8 * octets;
            const uint32_t fnx = 2u * g.nx, fny = 2u * g.ny;
            for (int it = (int)threadIdx.x; it < items; it += 64 * KS) {
                const int h = it % octets, r = it / octets;
                const int k = r & 7, vv = r >> 3;
                const uint32_t v = v0 + (uint32_t)vv;
                if (v >= V) continue;
                int x, y, z;
                vox_xyz(g, v, x, y, z);
                const uint32_t fv = ((2u * z + (k >> 2)) * fny + 2u * y + ((k >> 1) & 1)) * fnx + 2u * x + (k & 1);
                const size_t fo = (size_t)fv * cout_real + 8 * h;
                const uint4 sk = *(const uint4 *)(skip + fo);
                const uint32_t sw[4] = {sk.x, sk.y, sk.z, sk.w};
                uint32_t ow[4];
                const int j = vv >> 4, vl = vv & 15;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint16_t o[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int co = 8 * h + 2 * q + e;
                        const float av = s_a[(j * NT + (co >> 4)) * 4 + (vl & 3)][(vl >> 2) * 16 + (co & 15)];
                        o[e] = f2bf(av + bf2f((uint16_t)(sw[q] >> (16 * e))));
                    }
                    ow[q] = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
                }
                *(uint4 *)(yfine + fo) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
            }
            return;
        }
    }
    uint32_t vbase[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) vbase[j] = v0 + 16u * j;
    conv_store<NT, MT>(acc, vbase, V, m, grp, bias, cout_real, out, mode, proj, out2, g, skip, yfine);
}

template <int NT, int MT, int KS, bool CIN4>
__global__ void __launch_bounds__(KS > 1 ? 64 * KS : 256) k_conv_fwd(NetGeom g, const uint16_t *__restrict__ in, int cin,
                                                  const uint16_t *__restrict__ w,
                                                  const float *__restrict__ bias, int cout_real,
                                                  void *__restrict__ out, int mode,
                                                  const float *__restrict__ proj, float *__restrict__ out2,
                                                  const uint16_t *__restrict__ skip, uint16_t *__restrict__ yfine)
{
    conv_fwd_body<NT, MT, KS, CIN4>(g, in, cin, w, bias, cout_real, out, mode, proj, out2, skip, yfine,
                                    blockIdx.x, gridDim.x);
}

// Full-resolution convolution with its operands staged in LDS: a block
// computes a 16 x 4 x 4 voxel tile (wave w: y = w, M tiles z = 0..3) by 16
// output channels; the input tile with its one-voxel halo (18 x 6 x 6
// voxels) and the layer's weights are loaded once, so each input voxel is
// read from HBM/L2 about once instead of 27 times.  Requires nx % 16 == 0,
// ny % 4 == 0, nz % 4 == 0 and 16 output channels; cin 4 or 16.
template <bool CIN4>
__device__ __forceinline__ void conv_fwd_lds_body(const NetGeom &g, const uint16_t *__restrict__ in, int cin,
                                                  const uint16_t *__restrict__ w,
                                                  const float *__restrict__ bias, int cout_real,
                                                  void *__restrict__ out, int mode,
                                                  const float *__restrict__ proj, float *__restrict__ out2,
                                                  const uint16_t *__restrict__ skip,
                                                  uint16_t *__restrict__ yfine, uint32_t bid, uint32_t nblk)
{
    constexpr int CS = CIN4 ? 4 : 16;         // channels per voxel
    constexpr int HX = 18, HY = 6, HZ = 6;    // tile with halo
    __shared__ bf16x4 s_in[HX * HY * HZ * CS / 4];
    __shared__ bf16x4 s_w[27 * 16 * CS / 4];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wv = tid >> 6;
    const uint32_t tx = g.nx / 16u, ty = g.ny / 4u;
    const uint32_t t = xcd_tile(bid, nblk);  // one contiguous slab of tiles per XCD
    const uint32_t bx = t % tx, by = (t / tx) % ty, bz = t / (tx * ty);
    const int x0 = (int)bx * 16, y0 = (int)by * 4, z0 = (int)bz * 4;
    // stage the input tile (zeros or wrap-around outside the grid) and the
    // weights: every load of a thread is issued before its LDS stores
    constexpr int NIN = HX * HY * HZ * (CS / 4), NW = 27 * 16 * CS / 4;
    constexpr int UIN = (NIN + 255) / 256, UW = (NW + 255) / 256;
    bf16x4 vin[UIN], vw[UW];
#pragma unroll
    for (int u = 0; u < UIN; ++u) {
        const int q = (int)tid + 256 * u;
        vin[u] = bf16x4{0, 0, 0, 0};
        if (q < NIN) {
            const int vox = q / (CS / 4), part = q % (CS / 4);
            const int lx = vox % HX, ly = (vox / HX) % HY, lz = vox / (HX * HY);
            int x = x0 - 1 + lx, y = y0 - 1 + ly;
            const int z = z0 - 1 + lz;
            if (nb_in(g, x, y, z))
                vin[u] = *(const bf16x4 *)(in + ((size_t)((z * (int)g.ny + y) * (int)g.nx + x) * CS + part * 4));
        }
    }
#pragma unroll
    for (int u = 0; u < UW; ++u) {
        const int q = (int)tid + 256 * u;
        vw[u] = bf16x4{0, 0, 0, 0};
        if (q < NW) vw[u] = *(const bf16x4 *)(w + (size_t)q * 4);
    }
#pragma unroll
    for (int u = 0; u < UIN; ++u) {
        const int q = (int)tid + 256 * u;
        if (q < NIN) s_in[q] = vin[u];
    }
#pragma unroll
    for (int u = 0; u < UW; ++u) {
        const int q = (int)tid + 256 * u;
        if (q < NW) s_w[q] = vw[u];
    }
    __syncthreads();
    const uint32_t m = lane & 15u, grp = lane >> 4;
    f32x4 acc[4][1];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x4 zero4 = bf16x4{0, 0, 0, 0};
    if (CIN4) {
        // 32-wide steps of eight taps: lane group grp takes taps 8 st + 2 grp
        // and + 1 (four channels each); the padding taps 27..31 of the last
        // step read tap 26's operands and zero them
        for (int st = 0; st < 4; ++st) {
            bf16x4 al[4][2], bl[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int tap = 8 * st + 2 * (int)grp + e;
                const bool tok = tap < 27;
                const int tc = tok ? tap : 26;
                const int dz = tc / 9, dy = (tc / 3) % 3, dx = tc % 3;  // halo offsets 0..2
                bl[e] = tok ? s_w[tc * 16 + (int)m] : zero4;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bf16x4 a = s_in[((j + dz) * HY + ((int)wv + dy)) * HX + ((int)m + dx)];
                    al[j][e] = tok ? a : zero4;
                }
            }
            const s16x8 b = cat8(bl[0], bl[1]);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j][0] = mfma32(cat8(al[j][0], al[j][1]), b, acc[j][0]);
        }
    } else {
        // 32-wide steps of two taps: lane group grp reads channels
        // 8 (grp & 1) .. + 7 of tap 2 st + (grp >> 1); the padding tap 27
        // reads zeros
        const int half = (int)(grp & 1u), sub = (int)(grp >> 1);
        for (int st = 0; st < 14; ++st) {
            const int tap = 2 * st + sub;
            const bool tok = tap < 27;
            const int tc = tok ? tap : 26;
            const int dz = tc / 9, dy = (tc / 3) % 3, dx = tc % 3;
            const bf16x4 *wp = &s_w[(tc * 16 + (int)m) * 4 + 2 * half];
            const s16x8 b = tok ? cat8(wp[0], wp[1]) : cat8(zero4, zero4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bf16x4 *ap = &s_in[(((j + dz) * HY + ((int)wv + dy)) * HX + ((int)m + dx)) * 4 + 2 * half];
                const s16x8 a = tok ? cat8(ap[0], ap[1]) : cat8(zero4, zero4);
                acc[j][0] = mfma32(a, b, acc[j][0]);
            }
        }
    }
    (void)cin;
    const uint32_t V = g.nx * g.ny * g.nz;
    uint32_t vbase[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) vbase[j] = ((uint32_t)(z0 + j) * g.ny + (uint32_t)(y0 + (int)wv)) * g.nx + (uint32_t)x0;
    conv_store<1, 4>(acc, vbase, V, m, grp, bias, cout_real, out, mode, proj, out2, g, skip, yfine);
}

template <bool CIN4>
__global__ void __launch_bounds__(256) k_conv_fwd_lds(NetGeom g, const uint16_t *__restrict__ in, int cin,
                                                      const uint16_t *__restrict__ w,
                                                      const float *__restrict__ bias, int cout_real,
                                                      void *__restrict__ out, int mode,
                                                      const float *__restrict__ proj, float *__restrict__ out2,
                                                      const uint16_t *__restrict__ skip, uint16_t *__restrict__ yfine)
{
    conv_fwd_lds_body<CIN4>(g, in, cin, w, bias, cout_real, out, mode, proj, out2, skip, yfine, blockIdx.x,
                            gridDim.x);
}

template <int NT, bool CIN4>
static void conv_fwd_nt(hipStream_t s, const NetGeom &g, const uint16_t *in, int cin, const uint16_t *w,
                        const float *bias, int cout_real, void *out, int mode, const float *proj,
                        float *out2, const uint16_t *skip, uint16_t *yfine)
{
    const uint32_t V = g.nx * g.ny * g.nz;
    if (NT == 1 && V >= 65536u && g.nx % 16u == 0 && g.ny % 4u == 0 && g.nz % 4u == 0 &&
        (cin == 4 || cin == 16)) {
        const uint32_t blocks = (g.nx / 16u) * (g.ny / 4u) * (g.nz / 4u);
        hipLaunchKernelGGL((k_conv_fwd_lds<CIN4>), dim3(blocks), dim3(256), 0, s, g, in, cin, w, bias,
                           cout_real, out, mode, proj, out2, skip, yfine);
    } else if (V >= 65536u) {
        const uint32_t tiles = (V + 63u) / 64u;
        hipLaunchKernelGGL((k_conv_fwd<NT, 4, 1, CIN4>), dim3((tiles + 3u) / 4u), dim3(256), 0, s, g, in, cin,
                           w, bias, cout_real, out, mode, proj, out2, skip, yfine);
    } else if (V > CONV_SMALL_V) {
        // below 65536 voxels the 4 waves of a block split K for one 16-voxel
        // tile (and share an upsampling epilogue): four times the waves of
        // one tile per wave, which these latency-bound grids need
        const uint32_t tiles = (V + 15u) / 16u;
        hipLaunchKernelGGL((k_conv_fwd<NT, 1, 4, CIN4>), dim3(tiles), dim3(256), 0, s, g, in, cin, w, bias,
                           cout_real, out, mode, proj, out2, skip, yfine);
    } else if (cin >= 64) {
        // the longest K (27 x 64) of the small grids: 16 waves per tile
        const uint32_t tiles = (V + 15u) / 16u;
        hipLaunchKernelGGL((k_conv_fwd<NT, 1, 16, CIN4>), dim3(tiles), dim3(1024), 0, s, g, in, cin, w, bias,
                           cout_real, out, mode, proj, out2, skip, yfine);
    } else {
        const uint32_t tiles = (V + 15u) / 16u;
        hipLaunchKernelGGL((k_conv_fwd<NT, 1, CONV_KS_SMALL, CIN4>), dim3(tiles), dim3(64 * CONV_KS_SMALL), 0, s,
                           g, in, cin, w, bias, cout_real, out, mode, proj, out2, skip, yfine);
    }
}

// The kernel variants of conv_fwd_nt, in its order of choice.
#define CV_LDS 0
#define CV_BIG 1
#define CV_KS4 2
#define CV_KS16 3
#define CV_KS8 4

int conv_variant(const NetGeom &g, int cin, int cout_pad)
{
    const uint32_t V = g.nx * g.ny * g.nz;
    if (cout_pad == 16 && V >= 65536u && g.nx % 16u == 0 && g.ny % 4u == 0 && g.nz % 4u == 0 &&
        (cin == 4 || cin == 16))
        return CV_LDS;
    if (V >= 65536u) return CV_BIG;
    if (V > CONV_SMALL_V) return CV_KS4;
    if (cin >= 64) return CV_KS16;
    return CV_KS8;
}

uint32_t conv_variant_blocks(int variant, const NetGeom &g)
{
    const uint32_t V = g.nx * g.ny * g.nz;
    if (variant == CV_LDS) return (g.nx / 16u) * (g.ny / 4u) * (g.nz / 4u);
    if (variant == CV_BIG) return ((V + 63u) / 64u + 3u) / 4u;
    return (V + 15u) / 16u;
}

template <int NT, int MT, int KS, bool CIN4>
__global__ void __launch_bounds__(KS > 1 ? 64 * KS : 256) k_conv_fwd_multi(const ConvTask *__restrict__ t,
                                                                         MultiMap m)
{
    uint32_t k, bid, nblk;
    if (!multi_block(m, k, bid, nblk)) return;
    const ConvTask &T = t[k];
    conv_fwd_body<NT, MT, KS, CIN4>(T.g, T.in, T.cin, T.w, T.bias, T.cout_real, T.out, T.mode, T.proj, T.out2,
                                    T.skip, T.yfine, bid, nblk);
}

template <bool CIN4>
__global__ void __launch_bounds__(256) k_conv_fwd_lds_multi(const ConvTask *__restrict__ t, MultiMap m)
{
    uint32_t k, bid, nblk;
    if (!multi_block(m, k, bid, nblk)) return;
    const ConvTask &T = t[k];
    conv_fwd_lds_body<CIN4>(T.g, T.in, T.cin, T.w, T.bias, T.cout_real, T.out, T.mode, T.proj, T.out2,
                            T.skip, T.yfine, bid, nblk);
}

template <int NT, bool CIN4>
static void conv_multi_nt(hipStream_t s, int variant, const ConvTask *t, MultiMap m, uint32_t blocks)
{
    switch (variant) {
    case CV_LDS:
        if (NT == 1)
            hipLaunchKernelGGL((k_conv_fwd_lds_multi<CIN4>), dim3(blocks), dim3(256), 0, s, t, m);
        break;
    case CV_BIG:
        hipLaunchKernelGGL((k_conv_fwd_multi<NT, 4, 1, CIN4>), dim3(blocks), dim3(256), 0, s, t, m);
        break;
    case CV_KS4:
        hipLaunchKernelGGL((k_conv_fwd_multi<NT, 1, 4, CIN4>), dim3(blocks), dim3(256), 0, s, t, m);
        break;
    case CV_KS16:
        hipLaunchKernelGGL((k_conv_fwd_multi<NT, 1, 16, CIN4>), dim3(blocks), dim3(1024), 0, s, t, m);
        break;
    default:
        hipLaunchKernelGGL((k_conv_fwd_multi<NT, 1, CONV_KS_SMALL, CIN4>), dim3(blocks),
                           dim3(64 * CONV_KS_SMALL), 0, s, t, m);
    }
}

int launch_conv_fwd_multi(hipStream_t s, int variant, int cin, int cout_pad, const ConvTask *t, MultiMap m,
                          uint32_t blocks)
{
    if (!blocks) return 0;
    const bool c4 = cin == 4;
    if (!c4 && (cin % 16) != 0) return -1;
    if (variant == CV_LDS && cout_pad != 16) return -1;
#define CONV_NT_MULTI(NTV)                                                      \
    (c4 ? conv_multi_nt<NTV, true>(s, variant, t, m, blocks)                    \
        : conv_multi_nt<NTV, false>(s, variant, t, m, blocks))
    switch (cout_pad) {
    case 16: CONV_NT_MULTI(1); break;
    case 32: CONV_NT_MULTI(2); break;
    case 48: CONV_NT_MULTI(3); break;
    case 64: CONV_NT_MULTI(4); break;
    default: return -1;
    }
#undef CONV_NT_MULTI
    return 0;
}

int launch_conv_fwd(hipStream_t s, const NetGeom &g, const uint16_t *in, int cin, const uint16_t *w,
                    int cout_pad, const float *bias, int cout_real, void *out, int mode, const float *proj,
                    float *out2, const uint16_t *skip, uint16_t *yfine)
{
    const bool c4 = cin == 4;
    if (!c4 && (cin % 16) != 0) return -1;
    if (mode == NET_OUT_PROJ && (cout_pad != 16 || cout_real != 16 || !bias || !proj || !out2)) return -1;
    if (mode == NET_OUT_RELU_UP && (!skip || !yfine || (cout_real & 7) != 0)) return -1;
#define CONV_NT(NTV)                                                                                         \
    (c4 ? conv_fwd_nt<NTV, true>(s, g, in, cin, w, bias, cout_real, out, mode, proj, out2, skip, yfine)       \
        : conv_fwd_nt<NTV, false>(s, g, in, cin, w, bias, cout_real, out, mode, proj, out2, skip, yfine))
    switch (cout_pad) {
    case 16: CONV_NT(1); break;
    case 32: CONV_NT(2); break;
    case 48: CONV_NT(3); break;
    case 64: CONV_NT(4); break;
    default: return -1;
    }
#undef CONV_NT
    return 0;
}

// Backward of the pointwise head out[v] = sum_c h[v][c] w[c] + w[16]:
// dh[v][c] = dout[v] w[c], g[c] += sum_v dout[v] h[v][c], g[16] += sum_v
// dout[v].  One block per 1024 voxels, 16 voxels x 16 channels per pass.
__global__ void __launch_bounds__(256) k_proj_bwd(uint32_t V, const float *__restrict__ dout,
                                                  const uint16_t *__restrict__ h, const float *__restrict__ w,
                                                  float *__restrict__ dh, float *__restrict__ g)
{
    __shared__ float part[256], pb[16];
    const uint32_t c = threadIdx.x & 15u, vl = threadIdx.x >> 4;
    const uint32_t v0 = blockIdx.x * 1024u;
    const uint32_t ve = v0 + 1024u < V ? v0 + 1024u : V;
    const float wc = w[c];
    float sw = 0.f, sb = 0.f;
    for (uint32_t v = v0 + vl; v < ve; v += 16u) {
        const float d = dout[v];
        dh[(size_t)v * 16 + c] = d * wc;
        sw += d * bf2f(h[(size_t)v * 16 + c]);
        if (c == 0) sb += d;
    }
    part[threadIdx.x] = sw;
    if (c == 0) pb[vl] = sb;
    __syncthreads();
    if (threadIdx.x < 16) {
        float t = 0.f;
        for (int k = 0; k < 16; ++k) t += part[k * 16 + threadIdx.x];
        atomicAdd(g + threadIdx.x, t);
    } else if (threadIdx.x == 16) {
        float t = 0.f;
        for (int k = 0; k < 16; ++k) t += pb[k];
        atomicAdd(g + 16, t);
    }
}

void launch_proj_bwd(hipStream_t s, uint32_t V, const float *dout, const uint16_t *h, const float *w, float *dh,
                     float *g)
{
    hipLaunchKernelGGL(k_proj_bwd, dim3((V + 1023u) / 1024u), dim3(256), 0, s, V, dout, h, w, dh, g);
}

// ---------------------------------------------------------------------------
// Weight gradient dW[tap][co][ci] += sum_v dz[v][co] x[v + tap][ci] as
// MFMA tiles with M = 16 output channels, N = 16 input channels (CIN4: four
// taps of 4 channels) and K = 32 voxels per step.
//
// The contraction runs over voxels, so both operands are wanted eight voxels
// per lane while the activations are channels-last.  A block therefore stages
// a tile of 16 x 4 x 4 voxels transposed in LDS: dz as [channel][voxel], and x
// with its halo as three copies [channel][row][x], one for each x offset of a
// tap, so that every operand is one aligned 16-byte read.  The channel
// strides (528 and 1168 bytes) spread the 16 channels of a read over all 64
// banks.  Each of the four waves holds the 16 x 16 sums of seven taps (CIN4:
// two groups of four) over all of the block's tiles and adds them to dW with
// FP32 atomics at the end.  On the 48 x 48 x 96 grid a layer takes
// 9 to 27 us, the input layer 33, where one 2-byte load and one voxel division
// per operand element took 76 us on average and 107.
// ---------------------------------------------------------------------------
#define WT_X 16
#define WT_Y 4
#define WT_Z 4
#define WT_ROWS (WT_Y * WT_Z)                 // x rows of the tile
#define WT_HROWS ((WT_Y + 2) * (WT_Z + 2))    // x rows with the halo
#define WT_DZ_CH (WT_ROWS * WT_X + 8)         // channel strides, elements
#define WT_X_CH (WT_HROWS * WT_X + 8)
// Blocks a launch aims at: two per compute unit, and fewer for the input
// layer, whose 1,296 sums every block adds to (432 blocks took 60 us, 124
// blocks 33; the 16 to 16 channel layer with 6,912 sums 27 us with
// 432 blocks, 31 with 216).
#define WT_BLOCKS 512u
#define WT_BLOCKS_IN 128u

template <bool CIN4>
__global__ void __launch_bounds__(256) k_conv_wgrad(NetGeom g, const uint16_t *__restrict__ x, int cin,
                                                    const uint16_t *__restrict__ dz, int cout,
                                                    float *__restrict__ dw, int cin_real, uint32_t ntx,
                                                    uint32_t nty, uint32_t ntiles, uint32_t per,
                                                    uint32_t nci, uint32_t nchunk)
{
    constexpr int XC = CIN4 ? 4 : 16;   // staged input channels
    constexpr int NT = CIN4 ? 2 : 7;    // tap groups of a wave
    __shared__ __align__(16) uint16_t s_dz[16 * WT_DZ_CH];
    __shared__ __align__(16) uint16_t s_x[3 * XC * WT_X_CH];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t job = blockIdx.x;
    const uint32_t chunk = job % nchunk;
    job /= nchunk;
    const uint32_t cit = job % nci, cot = job / nci;
    const uint32_t m = lane & 15u, grp = lane >> 4;
    f32x4 acc[NT];
    int xoff[NT];  // this lane's B rows of each tap group: copy, channel, tap's y and z
    bool tok[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int q = (int)wave * NT + t;
        const int tap = CIN4 ? q * 4 + (int)(m >> 2) : q;
        const int ci = CIN4 ? (int)(m & 3u) : (int)m;
        tok[t] = tap < 27;
        const int tt = tok[t] ? tap : 13;
        xoff[t] = ((tt % 3) * XC + ci) * WT_X_CH + ((tt / 9) * (WT_Y + 2) + (tt / 3) % 3) * WT_X;
    }
    const uint32_t t1 = (chunk + 1u) * per < ntiles ? (chunk + 1u) * per : ntiles;
    for (uint32_t tile = chunk * per; tile < t1; ++tile) {
        const int bx = (int)(tile % ntx) * WT_X, by = (int)((tile / ntx) % nty) * WT_Y;
        const int bz = (int)(tile / (ntx * nty)) * WT_Z;
        __syncthreads();
        // dz: 256 voxels x 16 channels, 8 channels per item
        for (uint32_t i = tid; i < 2u * WT_ROWS * WT_X; i += 256u) {
            const uint32_t half = i & 1u, v = i >> 1;
            const int vx = bx + (int)(v % WT_X), vy = by + (int)((v / WT_X) % WT_Y);
            const int vz = bz + (int)(v / (WT_X * WT_Y));
            s16x8 q = {0, 0, 0, 0, 0, 0, 0, 0};
            if (vx < (int)g.nx && vy < (int)g.ny && vz < (int)g.nz)
                q = *(const s16x8 *)(dz + (size_t)((vz * (int)g.ny + vy) * (int)g.nx + vx) * cout + cot * 16u +
                                     half * 8u);
#pragma unroll
            for (int c = 0; c < 8; ++c) s_dz[(half * 8u + c) * WT_DZ_CH + v] = (uint16_t)q[c];
        }
        // x with its halo: 18 x 6 x 6 voxels
        constexpr uint32_t HV = (WT_X + 2) * WT_HROWS, PARTS = CIN4 ? 1u : 2u;
        for (uint32_t i = tid; i < HV * PARTS; i += 256u) {
            const uint32_t half = CIN4 ? 0u : i & 1u, v = CIN4 ? i : i >> 1;
            const uint32_t hx = v % (WT_X + 2), row = v / (WT_X + 2);
            int vx = bx + (int)hx - 1, vy = by + (int)(row % (WT_Y + 2)) - 1;
            const int vz = bz + (int)(row / (WT_Y + 2)) - 1;
            s16x8 q = {0, 0, 0, 0, 0, 0, 0, 0};
            // a tile may reach past the grid: only true neighbours of its voxels
            if (vx <= (int)g.nx && vy <= (int)g.ny && nb_in(g, vx, vy, vz)) {
                const uint16_t *p = x + (size_t)((vz * (int)g.ny + vy) * (int)g.nx + vx) * cin;
                if (CIN4) {
                    const bf16x4 h = *(const bf16x4 *)p;
                    q[0] = h[0], q[1] = h[1], q[2] = h[2], q[3] = h[3];
                } else {
                    q = *(const s16x8 *)(p + cit * 16u + half * 8u);
                }
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) {  // copy d holds x[t + d - 1] at t
                const int t = (int)hx - d;
                if (t < 0 || t >= WT_X) continue;
#pragma unroll
                for (int c = 0; c < (CIN4 ? 4 : 8); ++c)
                    s_x[((uint32_t)(d * XC) + half * 8u + c) * WT_X_CH + row * WT_X + t] = (uint16_t)q[c];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t ks = 0; ks < WT_ROWS / 2u; ++ks) {
            const uint32_t r = 2u * ks + (grp >> 1), x8 = 8u * (grp & 1u);
            const s16x8 a = *(const s16x8 *)(s_dz + m * WT_DZ_CH + r * WT_X + x8);
            const uint32_t rx = ((r / WT_Y) * (WT_Y + 2) + r % WT_Y) * WT_X + x8;
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[t] = mfma32(a, *(const s16x8 *)(s_x + xoff[t] + rx), acc[t]);
        }
    }
    // D[row = co tile row 4 grp + i][col = lane % 16]
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int q = (int)wave * NT + t;
        const int tap = CIN4 ? q * 4 + (int)(m >> 2) : q;
        const int ci = CIN4 ? (int)(m & 3u) : (int)(cit * 16u + m);
        if (!tok[t] || ci >= cin_real) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int co = (int)(cot * 16u + 4u * grp + (uint32_t)i);
            atomicAdd(dw + ((size_t)tap * cout + co) * cin_real + ci, acc[t][i]);
        }
    }
}

int launch_conv_wgrad(hipStream_t s, const NetGeom &g, const uint16_t *x, int cin, const uint16_t *dz,
                      int cout, float *dw, int cin_real)
{
    if (cout % 16 || (cin != 4 && cin % 16)) return -1;
    const uint32_t ntx = (g.nx + WT_X - 1) / WT_X, nty = (g.ny + WT_Y - 1) / WT_Y;
    const uint32_t ntiles = ntx * nty * ((g.nz + WT_Z - 1) / WT_Z);
    const uint32_t nci = cin == 4 ? 1u : (uint32_t)cin / 16u, pairs = nci * (uint32_t)cout / 16u;
    const uint32_t aim = cin == 4 ? WT_BLOCKS_IN : WT_BLOCKS;
    const uint32_t per = (ntiles * pairs + aim - 1u) / aim;
    const uint32_t nchunk = (ntiles + per - 1u) / per;
    if (cin == 4)
        hipLaunchKernelGGL(k_conv_wgrad<true>, dim3(nchunk * pairs), dim3(256), 0, s, g, x, cin, dz, cout, dw,
                           cin_real, ntx, nty, ntiles, per, nci, nchunk);
    else
        hipLaunchKernelGGL(k_conv_wgrad<false>, dim3(nchunk * pairs), dim3(256), 0, s, g, x, cin, dz, cout, dw,
                           cin_real, ntx, nty, ntiles, per, nci, nchunk);
    return 0;
}

// ---------------------------------------------------------------------------
// Elementwise kernels; fine grid g, coarse grid g/2 (even sizes).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void pool_fwd_body(const NetGeom &gc, const uint16_t *__restrict__ in, int c,
                                              uint16_t *__restrict__ out, uint32_t bid, uint32_t nblk)
{
    const uint32_t idx = xcd_tile(bid, nblk) * 256u + threadIdx.x;
    const uint32_t Vc = gc.nx * gc.ny * gc.nz;
    if (idx >= Vc * (uint32_t)c) return;
    const uint32_t vc = idx / (uint32_t)c, ch = idx % (uint32_t)c;
    int x, y, z;
    vox_xyz(gc, vc, x, y, z);
    const uint32_t fnx = 2u * gc.nx, fny = 2u * gc.ny;
    float sum = 0.f;
    for (int k = 0; k < 8; ++k) {
        const uint32_t fx = 2u * x + (k & 1), fy = 2u * y + ((k >> 1) & 1), fz = 2u * z + (k >> 2);
        sum += bf2f(in[((size_t)(fz * fny + fy) * fnx + fx) * c + ch]);
    }
    out[idx] = f2bf(0.125f * sum);
}

__global__ void __launch_bounds__(256) k_pool_fwd(NetGeom gc, const uint16_t *__restrict__ in, int c,
                                                  uint16_t *__restrict__ out)
{
    pool_fwd_body(gc, in, c, out, blockIdx.x, gridDim.x);
}

uint32_t pool_blocks(const NetGeom &gc, int c) { return (gc.nx * gc.ny * gc.nz * (uint32_t)c + 255u) / 256u; }

__global__ void __launch_bounds__(256) k_pool_fwd_multi(const PoolTask *__restrict__ t, MultiMap m)
{
    uint32_t k, bid, nblk;
    if (!multi_block(m, k, bid, nblk)) return;
    const PoolTask &T = t[k];
    pool_fwd_body(T.gc, T.in, T.c, T.out, bid, nblk);
}

void launch_pool_fwd_multi(hipStream_t s, const PoolTask *t, MultiMap m, uint32_t blocks)
{
    if (blocks) hipLaunchKernelGGL(k_pool_fwd_multi, dim3(blocks), dim3(256), 0, s, t, m);
}

void launch_pool_fwd(hipStream_t s, const NetGeom &gc, const uint16_t *in, int c, uint16_t *out)
{
    const uint32_t n = gc.nx * gc.ny * gc.nz * (uint32_t)c;
    hipLaunchKernelGGL(k_pool_fwd, dim3((n + 255u) / 256u), dim3(256), 0, s, gc, in, c, out);
}

// d_fine[v][c] += d_coarse[parent][c] / 8
__global__ void __launch_bounds__(256) k_pool_bwd(NetGeom gf, const float *__restrict__ dcoarse, int c,
                                                  float *__restrict__ dfine)
{
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    const uint32_t Vf = gf.nx * gf.ny * gf.nz;
    if (idx >= Vf * (uint32_t)c) return;
    const uint32_t vf = idx / (uint32_t)c, ch = idx % (uint32_t)c;
    int x, y, z;
    vox_xyz(gf, vf, x, y, z);
    const uint32_t cnx = gf.nx / 2u, cny = gf.ny / 2u;
    const size_t p = ((size_t)((z >> 1) * cny + (y >> 1)) * cnx + (x >> 1)) * c + ch;
    dfine[idx] += 0.125f * dcoarse[p];
}

void launch_pool_bwd(hipStream_t s, const NetGeom &gf, const float *dcoarse, int c, float *dfine)
{
    const uint32_t n = gf.nx * gf.ny * gf.nz * (uint32_t)c;
    hipLaunchKernelGGL(k_pool_bwd, dim3((n + 255u) / 256u), dim3(256), 0, s, gf, dcoarse, c, dfine);
}

// d_coarse[v][c] = sum of the 8 children's d_fine
__global__ void __launch_bounds__(256) k_up_bwd(NetGeom gc, const float *__restrict__ dfine, int c,
                                                float *__restrict__ dcoarse)
{
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    const uint32_t Vc = gc.nx * gc.ny * gc.nz;
    if (idx >= Vc * (uint32_t)c) return;
    const uint32_t vc = idx / (uint32_t)c, ch = idx % (uint32_t)c;
    int x, y, z;
    vox_xyz(gc, vc, x, y, z);
    const uint32_t fnx = 2u * gc.nx, fny = 2u * gc.ny;
    float sum = 0.f;
    for (int k = 0; k < 8; ++k) {
        const uint32_t fx = 2u * x + (k & 1), fy = 2u * y + ((k >> 1) & 1), fz = 2u * z + (k >> 2);
        sum += dfine[((size_t)(fz * fny + fy) * fnx + fx) * c + ch];
    }
    dcoarse[idx] = sum;
}

void launch_up_bwd(hipStream_t s, const NetGeom &gc, const float *dfine, int c, float *dcoarse)
{
    const uint32_t n = gc.nx * gc.ny * gc.nz * (uint32_t)c;
    hipLaunchKernelGGL(k_up_bwd, dim3((n + 255u) / 256u), dim3(256), 0, s, gc, dfine, c, dcoarse);
}

// dz = dy where the ReLU output y > 0, else 0, as BF16, and db[c] += sum_v
// dz[v][c] of the rounded values; C channels, a multiple of 4 up to 64.  A
// block takes `vpb` consecutive voxels, four channels per thread, and folds
// its sums in LDS.
__global__ void __launch_bounds__(256) k_relu_mask(uint32_t V, const float *__restrict__ dy,
                                                   const uint16_t *__restrict__ y, uint32_t C, uint32_t vpb,
                                                   uint16_t *__restrict__ dz, float *__restrict__ db)
{
    __shared__ float part[256][4];
    const uint32_t q = C / 4u, lanes = 256u / q;
    const uint32_t c4 = threadIdx.x % q, vl = threadIdx.x / q;
    const uint32_t v0 = blockIdx.x * vpb;
    const uint32_t ve = v0 + vpb < V ? v0 + vpb : V;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (vl < lanes)
        for (uint32_t v = v0 + vl; v < ve; v += lanes) {
            const size_t i = (size_t)v * C + 4u * c4;
            const f32x4 d = *(const f32x4 *)(dy + i);
            const bf16x4 a = *(const bf16x4 *)(y + i);
            bf16x4 r;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint16_t b = f2bf(bf2f((uint16_t)a[k]) > 0.f ? d[k] : 0.f);
                r[k] = (short)b;
                sum[k] += bf2f(b);
            }
            *(bf16x4 *)(dz + i) = r;
        }
#pragma unroll
    for (int k = 0; k < 4; ++k) part[threadIdx.x][k] = sum[k];
    __syncthreads();
    if (threadIdx.x < C) {
        float t = 0.f;
        for (uint32_t l = 0; l < lanes; ++l) t += part[l * q + threadIdx.x / 4u][threadIdx.x & 3u];
        atomicAdd(db + threadIdx.x, t);
    }
}

void launch_relu_mask(hipStream_t s, uint32_t V, const float *dy, const uint16_t *y, int c, uint16_t *dz,
                      float *db)
{
    // at least one voxel per thread, at most 512 blocks (two per compute unit)
    const uint32_t lanes = 256u / ((uint32_t)c / 4u);
    uint32_t vpb = (V + 511u) / 512u;
    if (vpb < lanes) vpb = lanes;
    hipLaunchKernelGGL(k_relu_mask, dim3((V + vpb - 1u) / vpb), dim3(256), 0, s, V, dy, y, (uint32_t)c, vpb, dz,
                       db);
}

// (an atomic add: passes of several networks may add to one dst)
__global__ void __launch_bounds__(256) k_add_and_clear(size_t n, float *__restrict__ src, float *__restrict__ dst)
{
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    atomicAdd(dst + i, src[i]);
    src[i] = 0.f;
}

void launch_add_and_clear(hipStream_t s, size_t n, float *src, float *dst)
{
    hipLaunchKernelGGL(k_add_and_clear, dim3((unsigned)((n + 255u) / 256u)), dim3(256), 0, s, n, src, dst);
}

// FP32 -> BF16 with channel padding: out[v][cpad] from in[v][c]
__global__ void __launch_bounds__(256) k_to_bf16_pad(uint32_t V, const float *__restrict__ in, int c,
                                                     int cpad, uint16_t *__restrict__ out)
{
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= V * (uint32_t)cpad) return;
    const uint32_t v = idx / (uint32_t)cpad, ch = idx % (uint32_t)cpad;
    out[idx] = (int)ch < c ? f2bf(in[(size_t)v * c + ch]) : (uint16_t)0;
}

void launch_to_bf16_pad(hipStream_t s, uint32_t V, const float *in, int c, int cpad, uint16_t *out)
{
    const uint32_t n = V * (uint32_t)cpad;
    hipLaunchKernelGGL(k_to_bf16_pad, dim3((n + 255u) / 256u), dim3(256), 0, s, V, in, c, cpad, out);
}

// Pack FP32 parameters (w[27][cout][cin] of each layer) into the BF16
// operand layouts: forward wf[27][cout_pad][cin_pad] and, for the data
// gradient (the adjoint: taps mirrored, channels swapped),
// wt[27][cin_pad2][cout_pad2] with wt[tap][ci][co] = w[26 - tap][co][ci].  One
// launch for all layers, and for the conversion of the network's input (in,
// rows of 3, to BF16 rows of 4; null: none), which the packing does not need:
// nine launches of 3 us took a quarter of a forward pass.
__global__ void __launch_bounds__(256) k_pack_weights(PackLayers p)
{
    int l = 0;
    while (l < p.n && blockIdx.x >= p.layer[l].blocks) ++l;
    const uint32_t b0 = l ? p.layer[l - 1].blocks : 0u;
    const uint32_t idx = (blockIdx.x - b0) * 256u + threadIdx.x;
    if (l == p.n) {
        if (idx >= p.V) return;
        const float *r = p.in + 3 * (size_t)idx;
        const bf16x4 o = {(short)f2bf(r[0]), (short)f2bf(r[1]), (short)f2bf(r[2]), 0};
        *(bf16x4 *)(p.in4 + 4 * (size_t)idx) = o;
        return;
    }
    const PackLayer &L = p.layer[l];
    const uint32_t cin = (uint32_t)L.cin, cout = (uint32_t)L.cout;
    if (idx < 27u * (uint32_t)L.cout_pad * (uint32_t)L.cin_pad) {
        const uint32_t ci = idx % (uint32_t)L.cin_pad;
        const uint32_t r = idx / (uint32_t)L.cin_pad;
        const uint32_t co = r % (uint32_t)L.cout_pad, tap = r / (uint32_t)L.cout_pad;
        L.wf[idx] = (ci < cin && co < cout) ? f2bf(L.w[((size_t)tap * cout + co) * cin + ci]) : (uint16_t)0;
    }
    if (L.wt && idx < 27u * (uint32_t)L.tout_pad * (uint32_t)L.tin_pad) {
        // wt layout [tap][new co = ci][new ci = co]
        const uint32_t nci = idx % (uint32_t)L.tin_pad;      // original output channel
        const uint32_t r = idx / (uint32_t)L.tin_pad;
        const uint32_t nco = r % (uint32_t)L.tout_pad, tap = r / (uint32_t)L.tout_pad;  // original input channel
        L.wt[idx] = (nci < cout && nco < cin) ? f2bf(L.w[((size_t)(26u - tap) * cout + nci) * cin + nco])
                                              : (uint16_t)0;
    }
}

void launch_pack_weights(hipStream_t s, PackLayers &p)
{
    uint32_t at = 0;
    for (int l = 0; l < p.n; ++l) {
        PackLayer &L = p.layer[l];
        uint32_t n = 27u * (uint32_t)L.cout_pad * (uint32_t)L.cin_pad;
        const uint32_t n2 = 27u * (uint32_t)L.tout_pad * (uint32_t)L.tin_pad;
        if (L.wt && n2 > n) n = n2;
        at += (n + 255u) / 256u;
        L.blocks = at;
    }
    if (p.in) at += (p.V + 255u) / 256u;
    hipLaunchKernelGGL(k_pack_weights, dim3(at), dim3(256), 0, s, p);
}
