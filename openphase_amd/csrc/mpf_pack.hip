// The state as concatenated lists (the raw .dat order, PhaseField::Write, src/PhaseField.cpp:
// 2340-2388): entry counts per block of cells and their running sums, and the packing of a range
// of cells into counts, grain indices, values and interface flags as the host receives them.
//
// Packed on the device, so that only the entries that exist cross to the host: 12 bytes each and 4
// per cell, instead of every stored slot (10 bytes each) for a host loop to pick from. At 128^3 with 16
// slots and 3.3 million entries a download took 94 ms, most of it that loop and the pages of its
// 335 MB of buffers; now 4.2 ms (a 1.2 ms step among them not counted). The transfer to pageable
// memory bounds it: the kernels take 50 us. Also the device checkpoints.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mpf_device.h"
#include "mpf_lists.h"

namespace mpf {

namespace {

constexpr int kPackBlock = 256;
constexpr int kPackPer = kPackCells / kPackBlock;  // cells of a thread

// Exclusive running sum of v over the block's threads; `total` the block's sum.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s_wave, uint32_t& total)
{
    const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;
    uint32_t sum = v;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(sum), k));
        if (lane >= k) sum += o;
    }
    if (lane == 63) s_wave[wave] = sum;
    __syncthreads();
    uint32_t before = sum - v;
    total = 0u;
#pragma unroll
    for (int w = 0; w < kPackBlock / 64; ++w) {
        before += w < wave ? s_wave[w] : 0u;
        total += s_wave[w];
    }
    __syncthreads();
    return before;
}

// offset[b + 1] = entries of the cells of block b.
template <typename TV>
__global__ __launch_bounds__(kPackBlock) void pack_count_kernel(const uint8_t* __restrict__ cnt, int64_t ncells,
                                                                int64_t* __restrict__ offset)
{
    __shared__ uint32_t s_wave[kPackBlock / 64];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kPackCells;
    uint32_t n = 0u;
    for (int k = static_cast<int>(threadIdx.x); k < kPackCells; k += kPackBlock)
        if (base + k < ncells) n += static_cast<uint32_t>(ListCode<TV>::count(cnt[base + k]));
    uint32_t total;
    (void)block_scan(n, s_wave, total);
    if (threadIdx.x == 0) offset[blockIdx.x + 1] = total;
}

// offset[1 .. blocks] to running sums; offset[0] = 0. One block.
__global__ __launch_bounds__(kPackBlock) void pack_scan_kernel(int64_t* offset, int64_t blocks)
{
    __shared__ uint32_t s_wave[kPackBlock / 64];
    int64_t done = 0;
    if (threadIdx.x == 0) offset[0] = 0;
    for (int64_t i0 = 1; i0 <= blocks; i0 += kPackBlock) {
        const int64_t i = i0 + threadIdx.x;
        const uint32_t v = i <= blocks ? static_cast<uint32_t>(offset[i]) : 0u;
        uint32_t total;
        const uint32_t before = block_scan(v, s_wave, total);
        if (i <= blocks) offset[i] = done + before + v;
        done += total;
    }
}

// Packs the cells of blocks first .. first + gridDim.x - 1: count[c], flag[c] (either may be null), and
// the entries from position offset[b] - offset[first] on.
template <typename TV>
__global__ __launch_bounds__(kPackBlock) void pack_write_kernel(const StepArgs A, const int64_t* __restrict__ offset, int64_t first,
                                                                int32_t* __restrict__ count, int8_t* __restrict__ flag,
                                                                int32_t* __restrict__ index, double* __restrict__ value)
{
    __shared__ uint32_t s_wave[kPackBlock / 64];
    const int64_t N = A.ncells, b = first + blockIdx.x;
    int64_t at = offset[b] - offset[first];
    for (int k = 0; k < kPackPer; ++k) {
        const int64_t c = b * kPackCells + k * kPackBlock + threadIdx.x;
        const bool in = c < N;
        const uint8_t code = in ? A.cnt_in[c] : 0;
        const int n = ListCode<TV>::count(code), imp = ListCode<TV>::implicit(code);
        uint32_t total;
        int64_t to = at + block_scan(static_cast<uint32_t>(n), s_wave, total);
        at += total;
        if (!in) continue;
        const int64_t out = c - first * kPackCells;
        if (count) count[out] = n;
        if (flag) {
            // flag 2: more than one entry; flag 1: such a cell in the box
            uint32_t codes[7];
            flag[out] = n > 1 ? 2 : (load_codes<TV>(A, make_box(A, c), code, codes) ? 1 : 0);
        }
        double others = 0.0;
        for (int q = 0; q < n; ++q) {
            const double v = q != imp ? static_cast<double>(load_val<TV>(A.val_in, static_cast<int64_t>(q) * N + c)) : 0.0;
            if (q != imp) others += v;
            if (index) index[to + q] = A.id_in[static_cast<int64_t>(q) * N + c];
            if (value) value[to + q] = v;
        }
        // FP32: the implicit entry is 1 - the sum of the others
        if (value && imp >= 0 && imp < n) value[to + imp] = 1.0 - others;
    }
}

// Checkpoints (mpf_save_state, mpf_restore_state) in one launch each instead of eight copies, which
// small domains feel most: 6 us of kernel for a domain of 128^2 to 512^2. 64 such domains restored and
// stepped 40 times took 23.1 ms and take 20.1 ms; 512^2 in FP64 with 20 steps 1.11 and 1.05 ms.

// A saved state into the context: counts, the entries in use, grain arrays. Slots a cell does not use
// are never read, so they are left: at 256^3 with 16 slots a restore takes 0.26 ms, a copy of every slot
// (the save) 1.1 ms.
template <typename TV>
__global__ __launch_bounds__(256) void restore_kernel(const StateCopy S)
{
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (c < S.ncells) {
        const uint8_t code = S.src.cnt[c];
        S.dst.cnt[c] = code;
        const int n = min(ListCode<TV>::count(code), S.slots);
        for (int s = 0; s < n; ++s) {
            const int64_t at = static_cast<int64_t>(s) * S.ncells + c;
            S.dst.id[at] = S.src.id[at];
            static_cast<TV*>(S.dst.val)[at] = static_cast<const TV*>(S.src.val)[at];
        }
    }
    if (c < S.ngrains) {
        S.dst.volume[c] = S.src.volume[c];
        S.dst.maxvolume[c] = S.src.maxvolume[c];
        S.dst.vr[c] = S.src.vr[c];
        S.dst.exist[c] = S.src.exist[c];
        S.dst.stage[c] = S.src.stage[c];
    }
}

// The context's state into a checkpoint, every slot.
__global__ __launch_bounds__(256) void save_kernel(const StateCopy S, int value_bytes)
{
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, stride = static_cast<int64_t>(gridDim.x) * 256;
    auto copy = [&](void* dst, const void* src, int64_t bytes) {
        const int64_t n = bytes / 16;
        for (int64_t i = i0; i < n; i += stride) static_cast<uint4*>(dst)[i] = static_cast<const uint4*>(src)[i];
        for (int64_t i = 16 * n + i0; i < bytes; i += stride) static_cast<uint8_t*>(dst)[i] = static_cast<const uint8_t*>(src)[i];
    };
    copy(S.dst.cnt, S.src.cnt, S.ncells);
    copy(S.dst.id, S.src.id, S.ncells * S.slots * 2);
    copy(S.dst.val, S.src.val, S.ncells * S.slots * value_bytes);
    for (int64_t g = i0; g < S.ngrains; g += stride) {
        S.dst.volume[g] = S.src.volume[g];
        S.dst.maxvolume[g] = S.src.maxvolume[g];
        S.dst.vr[g] = S.src.vr[g];
        S.dst.exist[g] = S.src.exist[g];
        S.dst.stage[g] = S.src.stage[g];
    }
}

}  // namespace

int launch_restore(const StateCopy& a, bool fp32, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t n = a.ncells > a.ngrains ? a.ncells : a.ngrains;
    const dim3 grid(static_cast<unsigned>((n + 255) / 256));
    if (fp32) hipLaunchKernelGGL((restore_kernel<float>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((restore_kernel<double>), grid, dim3(256), 0, s, a);
    return static_cast<int>(hipGetLastError());
}

int launch_save(const StateCopy& a, bool fp32, void* stream)
{
    const int64_t n = a.ncells * a.slots / 1024 + 1;
    const dim3 grid(static_cast<unsigned>(n < 16384 ? n : 16384));
    hipLaunchKernelGGL(save_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), a, fp32 ? 4 : 8);
    return static_cast<int>(hipGetLastError());
}

int64_t pack_blocks(int64_t ncells) { return (ncells + kPackCells - 1) / kPackCells; }

int launch_pack_offsets(const uint8_t* cnt, int64_t ncells, bool fp32, int64_t* offset, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t nb = pack_blocks(ncells);
    const dim3 grid(static_cast<unsigned>(nb));
    if (fp32) hipLaunchKernelGGL((pack_count_kernel<float>), grid, dim3(kPackBlock), 0, s, cnt, ncells, offset);
    else hipLaunchKernelGGL((pack_count_kernel<double>), grid, dim3(kPackBlock), 0, s, cnt, ncells, offset);
    hipLaunchKernelGGL(pack_scan_kernel, dim3(1), dim3(kPackBlock), 0, s, offset, nb);
    return static_cast<int>(hipGetLastError());
}

int launch_pack(const StepArgs& a, bool fp32, const int64_t* offset, int64_t first, int64_t blocks, int32_t* count, int8_t* flag,
                int32_t* index, double* value, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(blocks));
    if (fp32) hipLaunchKernelGGL((pack_write_kernel<float>), grid, dim3(kPackBlock), 0, s, a, offset, first, count, flag, index, value);
    else hipLaunchKernelGGL((pack_write_kernel<double>), grid, dim3(kPackBlock), 0, s, a, offset, first, count, flag, index, value);
    return static_cast<int>(hipGetLastError());
}

}  // namespace mpf
