// Z-Sobol sample generation on the device (the sampler of Sources/libgonzales/Sampler/
// ZSobolSampler.swift, driven per path as Core/Tile.swift:28-33 does: startPixelSample, then a
// fixed sequence of get1D/get2D/get3D calls). One lane per (pixel, sample index).
#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "gz_internal.h"
#include "zsobol_device.h"

namespace gz {

const uint32_t *sobol_table();  // sobol_table.cpp

constexpr int kZsBlock = 256;
constexpr int kMaxCalls = 64;

struct CallPattern {
        int8_t calls[kMaxCalls];
        int32_t n;
        int32_t stride;
};

// The samples of a block's lanes on their way out, up to kStageDims dimensions at a time. In the layout of
// one row per sample a lane's values lie a row apart from its neighbours': written one by one, each store
// touched 26 lines for 256 bytes (13 dimensions), and that, not the digits, bound the kernel: 640 x 360
// pixels x 16 samples x 13 dimensions, 192 MB, took 256 us, and 277 with the grouped digits alone. Through LDS
// the block writes its rows in one run: 112 us with both (1.7 TB/s; now the table loads and integer work).
constexpr int kStageDims = 16;

struct Out {
        float *out;
        int64_t n, block, i;  // samples in all, the block's first, the lane's own
        int stride, soa;
        float *stage;
        int at, from;  // dimensions staged, the row's dimension of the first of them

        __device__ __forceinline__ void put(float v, int k) {
                if (soa) {
                        if (i < n) out[(int64_t)k * n + i] = v;
                        return;
                }
                const int width = stride - from < kStageDims ? stride - from : kStageDims;
                stage[threadIdx.x * width + at] = v;
                if (++at == width) flush(width);
        }
        __device__ __forceinline__ void flush(int width) {
                __syncthreads();
                const int rows = n - block < kZsBlock ? (int)(n - block) : kZsBlock;
                if (width == stride) {
                        float *o = out + block * stride;
                        for (int f = threadIdx.x; f < rows * width; f += kZsBlock) o[f] = stage[f];
                } else {
                        for (int f = threadIdx.x; f < rows * width; f += kZsBlock) {
                                const int row = f / width;
                                out[(block + row) * stride + from + (f - row * width)] = stage[f];
                        }
                }
                __syncthreads();
                from += width;
                at = 0;
        }
};

// mode 0: explicit (px, py, index) lists; mode 1: a tile x0..x0+w, y0..y0+h, spp samples per
// pixel, sample i = pixel (i / spp) in row-major order, index i % spp (Tile.swift:28-29 order).
// Lanes past n compute the last sample again and write nothing.
template <int kMode>
__global__ __launch_bounds__(kZsBlock) void k_zsobol(ZSobolParams p, const uint32_t *__restrict__ table,
                                                     const int32_t *__restrict__ pxs, const int32_t *__restrict__ pys,
                                                     const int64_t *__restrict__ idxs, int32_t x0, int32_t y0,
                                                     int32_t w, int32_t spp, int64_t n, int32_t startDim,
                                                     CallPattern pat, float *__restrict__ out, int32_t soa) {
        __shared__ float stage[kStageDims * kZsBlock];
        const int64_t block = (int64_t)blockIdx.x * kZsBlock, i = block + threadIdx.x, j = i < n ? i : n - 1;
        Out o{out, n, block, i, pat.stride, soa, stage, 0, 0};
        int32_t px, py;
        int64_t index;
        if (kMode == 0) {
                px = pxs[j];
                py = pys[j];
                index = idxs[j];
        } else {
                const int64_t pix = j / spp;
                index = j % spp;
                px = x0 + (int32_t)(pix % w);
                py = y0 + (int32_t)(pix / w);
        }
        ZSobolState z = zs_start(p, px, py, index, startDim);
        int k = 0;
        for (int c = 0; c < pat.n; ++c) {
                const int8_t kind = pat.calls[c];
                if (kind == 1) {
                        o.put(zs_get1d(p, z, table), k++);
                } else if (kind == 2) {
                        float a, b;
                        zs_get2d(p, z, table, a, b);
                        o.put(a, k++);
                        o.put(b, k++);
                } else {
                        float a, b, cc;
                        zs_get3d(p, z, table, a, b, cc);
                        o.put(a, k++);
                        o.put(b, k++);
                        o.put(cc, k++);
                }
        }
}

// The tile form for spp = 2^log2spp and indexes below 2^32 (grouped_tile). The digits above the sample
// index are the pixel's own: a group of up to 16 lanes (a DPP row) holds samples of one pixel, so its
// lanes compute one pixel digit each (in turn where the group is smaller) and OR them, and every lane
// adds only the digits of its sample index: 13 digits a call, two 32-bit multiplies each, become 3 to 4
// for 16 samples a pixel. (Lanes past n are whole groups: n is a multiple of the samples per pixel.)
__global__ __launch_bounds__(kZsBlock) void k_zsobol_grouped(ZSobolParams p, const uint32_t *__restrict__ table,
                                                             int32_t x0, int32_t y0, uint32_t w, int64_t n,
                                                             int32_t startDim, CallPattern pat,
                                                             float *__restrict__ out, int32_t soa) {
        __shared__ float stage[kStageDims * kZsBlock];
        const int64_t block = (int64_t)blockIdx.x * kZsBlock, i = block + threadIdx.x;
        Out o{out, n, block, i, pat.stride, soa, stage, 0, 0};
        const int L = p.log2spp, odd = L & 1, lg = L < 4 ? L : 4, group = 1 << lg;
        const uint32_t pix = (uint32_t)(i >> L), row = pix / w;
        const uint32_t morton = ((uint32_t)zs_morton2((uint32_t)x0 + (pix - row * w), (uint32_t)y0 + row) << L) |
                                ((uint32_t)i & ((1u << L) - 1u));
        const int own = (int)(threadIdx.x & (unsigned)(group - 1));
        const int firstPixelDigit = (L + 1) >> 1;
        int dim = startDim, k = 0;
        for (int c = 0; c < pat.n; ++c) {
                const int kind = pat.calls[c];
                const uint32_t mix = zs_dim_mix(dim);
                uint32_t idx = 0;
                for (int d = firstPixelDigit + own; d < p.nBase4Digits; d += group) {
                        const int shift = 2 * d - odd;
                        idx |= zs_digit32(morton, shift, mix) << shift;
                }
                if (lg > 0) idx |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)idx, 0xB1, 15, 15, false);   // lane ^ 1
                if (lg > 1) idx |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)idx, 0x4E, 15, 15, false);   // lane ^ 2
                if (lg > 2) idx |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)idx, 0x141, 15, 15, false);  // half row mirrored
                if (lg > 3) idx |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)idx, 0x140, 15, 15, false);  // row mirrored
                for (int d = odd; d < firstPixelDigit && d < p.nBase4Digits; ++d) {
                        const int shift = 2 * d - odd;
                        idx |= zs_digit32(morton, shift, mix) << shift;
                }
                if (odd) idx |= (morton ^ zs_mix_bits((uint64_t)((morton >> 1) ^ mix))) & 1u;
                // the seeds and the dimension's wrap of zs_get1d, zs_get2d and zs_get3d
                const uint32_t seeds[3] = {zs_hash(p, dim), 0u, zs_hash(p, dim + 2)};
                if (dim + kind - 1 >= kSobolDims) dim = 2;
                for (int q = 0; q < kind; ++q, ++k) o.put(zs_sobol32(idx, dim + q, seeds[q], table), k);
                dim += kind;
        }
}

// Whether a tile takes k_zsobol_grouped.
static bool grouped_tile(const GzZSobolParams &p, int64_t x0, int64_t y0, int64_t w, int64_t h, int64_t spp, int64_t n) {
        const int L = p.log2SamplesPerPixel;
        if (L > 16 || spp != (int64_t)1 << L || p.nBase4Digits > 16 || n >= (int64_t)1 << 32) return false;
        const int64_t side = std::max(x0 + w, y0 + h);  // every coordinate is below it
        return side <= (int64_t)1 << ((32 - L) / 2);
}

static std::mutex g_table_mu;
static uint32_t *g_dev_table[64] = {nullptr};

// The byte table of the 1024 x 52 matrix table (zsobol_device.h), on the host.
static std::vector<uint32_t> byte_table() {
        const uint32_t *cols = sobol_table();
        std::vector<uint32_t> t(kSobolByteTableWords, 0u);
        for (int d = 0; d < kSobolDims; ++d)
                for (int k = 0; k < kSobolBytes; ++k)
                        for (int v = 0; v < 256; ++v) {
                                uint32_t acc = 0;
                                for (int j = 0; j < 8; ++j) {
                                        const int c = 8 * k + j;
                                        if (((v >> j) & 1) && c < kSobolCols) acc ^= cols[d * kSobolCols + c];
                                }
                                t[((size_t)d * kSobolBytes + k) * 256 + v] = acc;
                        }
        return t;
}

// Device copy of the matrices in their byte-table form (7 MiB), made once per device.
const uint32_t *device_sobol_table() {
        int dev = 0;
        if (!hip_ok(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
        if (dev < 0 || dev >= 64) {
                set_error("device ordinal %d out of range", dev);
                return nullptr;
        }
        std::lock_guard<std::mutex> lock(g_table_mu);
        if (!g_dev_table[dev]) {
                uint32_t *d = nullptr;
                const size_t bytes = sizeof(uint32_t) * kSobolByteTableWords;
                if (!hip_ok(hipMalloc((void **)&d, bytes), "hipMalloc(sobol table)")) return nullptr;
                const std::vector<uint32_t> host = byte_table();
                if (!hip_ok(hipMemcpy(d, host.data(), bytes, hipMemcpyHostToDevice), "upload sobol table")) {
                        (void)hipFree(d);
                        return nullptr;
                }
                g_dev_table[dev] = d;
        }
        return g_dev_table[dev];
}

static bool make_pattern(const int8_t *pattern, int32_t nCalls, CallPattern &pat) {
        if (nCalls < 0 || nCalls > kMaxCalls || (nCalls > 0 && !pattern)) {
                set_error("call pattern: %d calls (0..%d allowed)", nCalls, kMaxCalls);
                return false;
        }
        std::memset(&pat, 0, sizeof pat);
        pat.n = nCalls;
        for (int c = 0; c < nCalls; ++c) {
                if (pattern[c] < 1 || pattern[c] > 3) {
                        set_error("call pattern entry %d is %d (must be 1, 2 or 3)", c, (int)pattern[c]);
                        return false;
                }
                pat.calls[c] = pattern[c];
                pat.stride += pattern[c];
        }
        return true;
}

static bool check_params(const GzZSobolParams *params, int32_t startDim) {
        if (!params) {
                set_error("null sampler parameters");
                return false;
        }
        if (params->log2SamplesPerPixel < 0 || params->log2SamplesPerPixel > 64 || params->nBase4Digits < 0 ||
            params->nBase4Digits > 64 || params->seed < 0) {
                set_error("sampler parameters out of range");
                return false;
        }
        if (startDim < 0 || startDim >= kSobolDims) {
                set_error("start dimension %d outside [0, %d)", startDim, kSobolDims);
                return false;
        }
        return true;
}

}  // namespace gz

using namespace gz;

// ZSobolSampler.init (ZSobolSampler.swift:114-122).
extern "C" int gz_zsobol_params(int64_t samplesPerPixel, int64_t resX, int64_t resY, int64_t seed,
                                GzZSobolParams *out) {
        clear_error();
        if (!out || seed < 0 || resX < 0 || resY < 0) {
                set_error("gz_zsobol_params: bad arguments");
                return GZ_E_INVALID;
        }
        const int tzSpp = samplesPerPixel == 0 ? 64 : __builtin_ctzll((unsigned long long)samplesPerPixel);
        int64_t r = resX > resY ? resX : resY;
        r -= 1;
        r |= r >> 1;
        r |= r >> 2;
        r |= r >> 4;
        r |= r >> 8;
        r |= r >> 16;
        r += 1;
        const int tzRes = r == 0 ? 64 : __builtin_ctzll((unsigned long long)r);
        out->seed = seed;
        out->log2SamplesPerPixel = tzSpp;
        out->nBase4Digits = tzRes + (tzSpp + 1) / 2;
        return GZ_OK;
}

extern "C" int gz_zsobol_samples_device(const GzZSobolParams *params, const int32_t *d_px, const int32_t *d_py,
                                        const int64_t *d_sampleIndex, int64_t count, int32_t startDim,
                                        const int8_t *pattern, int32_t nCalls, float *d_out, int32_t layout,
                                        void *stream) {
        clear_error();
        if (!check_params(params, startDim)) return GZ_E_INVALID;
        CallPattern pat;
        if (!make_pattern(pattern, nCalls, pat)) return GZ_E_INVALID;
        if (count < 0 || (count > 0 && (!d_px || !d_py || !d_sampleIndex || !d_out))) {
                set_error("gz_zsobol_samples_device: bad buffers");
                return GZ_E_INVALID;
        }
        if (count == 0 || pat.n == 0) return GZ_OK;
        const uint32_t *table = device_sobol_table();
        if (!table) return GZ_E_HIP;
        ZSobolParams p{params->seed, params->log2SamplesPerPixel, params->nBase4Digits};
        hipLaunchKernelGGL(k_zsobol<0>, dim3((unsigned)((count + kZsBlock - 1) / kZsBlock)), dim3(kZsBlock), 0,
                           static_cast<hipStream_t>(stream), p, table, d_px, d_py, d_sampleIndex, 0, 0, 1, 1, count,
                           startDim, pat, d_out, layout ? 1 : 0);
        return hip_ok(hipGetLastError(), "zsobol launch") ? GZ_OK : GZ_E_HIP;
}

extern "C" int gz_zsobol_tile_device(const GzZSobolParams *params, int32_t x0, int32_t y0, int32_t width,
                                     int32_t height, int32_t spp, int32_t startDim, const int8_t *pattern,
                                     int32_t nCalls, float *d_out, int32_t layout, void *stream) {
        clear_error();
        if (!check_params(params, startDim)) return GZ_E_INVALID;
        CallPattern pat;
        if (!make_pattern(pattern, nCalls, pat)) return GZ_E_INVALID;
        if (width < 0 || height < 0 || spp < 0 || x0 < 0 || y0 < 0) {
                set_error("gz_zsobol_tile_device: negative tile size");
                return GZ_E_INVALID;
        }
        const int64_t count = (int64_t)width * height * spp;
        if (count == 0 || pat.n == 0) return GZ_OK;
        if (!d_out) {
                set_error("gz_zsobol_tile_device: null output");
                return GZ_E_INVALID;
        }
        const uint32_t *table = device_sobol_table();
        if (!table) return GZ_E_HIP;
        ZSobolParams p{params->seed, params->log2SamplesPerPixel, params->nBase4Digits};
        if (grouped_tile(*params, x0, y0, width, height, spp, count)) {
                hipLaunchKernelGGL(k_zsobol_grouped, dim3((unsigned)((count + kZsBlock - 1) / kZsBlock)), dim3(kZsBlock), 0,
                                   static_cast<hipStream_t>(stream), p, table, x0, y0, (uint32_t)width, count, startDim, pat,
                                   d_out, layout ? 1 : 0);
                return hip_ok(hipGetLastError(), "zsobol launch") ? GZ_OK : GZ_E_HIP;
        }
        hipLaunchKernelGGL(k_zsobol<1>, dim3((unsigned)((count + kZsBlock - 1) / kZsBlock)), dim3(kZsBlock), 0,
                           static_cast<hipStream_t>(stream), p, table, nullptr, nullptr, nullptr, x0, y0, width, spp,
                           count, startDim, pat, d_out, layout ? 1 : 0);
        return hip_ok(hipGetLastError(), "zsobol launch") ? GZ_OK : GZ_E_HIP;
}
