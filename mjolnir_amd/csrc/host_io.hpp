// Transfers between the caller's arrays and the device state through pinned host memory: kernels
// pack the wanted double4 arrays into x, y, z triples there (downloads) or take triples from
// there (uploads), and the host copies between it and the caller's arrays.
//
// A transfer is bound by the host: one launch and one wait for a small system (three synchronous
// copies through the runtime's staging before, about 20 us each, then a conversion loop over a
// temporary), and the first touch of the caller's pages for a large one.  Measured with positions,
// velocities and forces: a replica of about 600 beads 64 -> 16 us a call, the 512 replicas of an
// ensemble one after the other 33 -> 9.8 ms.
#pragma once
#include "device_common.hpp"

#include <cstring>

namespace mjg
{
struct PackArgs
{
    const double4* src[3];
};

// out[a][3 i + c] = component c of src[a][first + i], i < n, one array per blockIdx.y: consecutive
// threads write consecutive words, so a wave's 512 bytes leave as whole lines
static __global__ void __launch_bounds__(256)
k_pack_xyz(PackArgs a, uint32_t first, uint32_t n, double* __restrict__ out)
{
    const double* s = reinterpret_cast<const double*>(a.src[blockIdx.y] + first);
    double* o = out + (size_t)blockIdx.y * 3 * n;
    for(uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < 3 * n; t += gridDim.x * blockDim.x)
    {
        o[t] = s[4 * (size_t)(t / 3) + t % 3];
    }
}

// to[first + i] = the triple in[3 i ..], wrapped into the box as System::initialize wraps positions
// (System.hpp:63-67, BoundaryCondition.hpp:93-102); a box that is not periodic leaves it as it is
static __global__ void __launch_bounds__(256)
k_unpack_xyz(const double* __restrict__ in, uint32_t first, uint32_t n, Box box, double4* __restrict__ to)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) {return;}
    double x = in[3 * (size_t)i], y = in[3 * (size_t)i + 1], z = in[3 * (size_t)i + 2];
    adjust_position(box, x, y, z);
    to[first + i] = make_double4(x, y, z, 0.0);
}

// Two pinned halves: while the host works on one, the device works on the other.  One owner (an
// engine or a batch), used by the one host thread that drives it; both halves are idle between calls.
class StateTransfer
{
  public:
    // largest half: holds the state of the largest replica (2048 particles, 144 KiB), and a chunk's
    // launch and wait are small beside its copy (about 10 against 50 us); pinning 1 MiB halves
    // instead made an engine 4 ms slower to create
    static constexpr size_t kHalfMax = size_t(1) << 18;

    ~StateTransfer()
    {
        for(hipEvent_t e : ev_) {if(e) {(void)hipEventDestroy(e);}}
        if(pin_) {(void)hipHostFree(pin_);}
    }
    // room for the whole state of n particles in one half, up to kHalfMax bytes
    hipError_t create(size_t n)
    {
        half_ = std::min(kHalfMax, 9 * n * sizeof(double));
        hipError_t e = hipHostMalloc(&pin_, 2 * half_, hipHostMallocDefault);
        if(e != hipSuccess) {(void)hipGetLastError(); pin_ = nullptr; return e;}
        for(auto& v : ev_)
        {
            e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
            if(e != hipSuccess) {return e;}
        }
        return hipSuccess;
    }
    // the arrays src[k] with a destination dst[k] (3 n doubles each), in the order of the stream
    hipError_t download(const double4* const (&src)[3], double* const (&dst)[3], size_t n, hipStream_t stream)
    {
        PackArgs a{};
        double* to[3];
        uint32_t m = 0;
        for(int k = 0; k < 3; ++k) {if(dst[k]) {a.src[m] = src[k]; to[m] = dst[k]; ++m;}}
        if(m == 0 || n == 0) {return hipSuccess;}
        const size_t per = half_ / (3 * sizeof(double) * m);       // particles per chunk
        const size_t chunks = (n + per - 1) / per;
        auto size_of = [&](size_t c) {return std::min(per, n - c * per);};
        auto fill = [&](size_t c) -> hipError_t {
            const uint32_t k = (uint32_t)size_of(c);
            double* half = reinterpret_cast<double*>(static_cast<char*>(pin_) + (c & 1) * half_);
            const uint32_t blocks = std::min<uint32_t>((3 * k + 255) / 256, 256);
            hipLaunchKernelGGL(k_pack_xyz, dim3(blocks, m), dim3(256), 0, stream, a, (uint32_t)(c * per), k, half);
            const hipError_t e = hipGetLastError();
            // a single chunk is waited for on the stream itself
            return (e != hipSuccess || chunks == 1) ? e : hipEventRecord(ev_[c & 1], stream);
        };
        for(size_t c = 0; c < std::min<size_t>(2, chunks); ++c)
        {
            const hipError_t e = fill(c);
            if(e != hipSuccess) {return e;}
        }
        for(size_t c = 0; c < chunks; ++c)
        {
            hipError_t e = (chunks == 1) ? hipStreamSynchronize(stream) : hipEventSynchronize(ev_[c & 1]);
            if(e != hipSuccess) {return e;}
            const size_t k = size_of(c);
            const double* half = reinterpret_cast<const double*>(static_cast<const char*>(pin_) + (c & 1) * half_);
            for(uint32_t q = 0; q < m; ++q)
            {
                std::memcpy(to[q] + 3 * c * per, half + (size_t)q * 3 * k, 3 * k * sizeof(double));
            }
            if(c + 2 < chunks)
            {
                e = fill(c + 2);
                if(e != hipSuccess) {return e;}
            }
        }
        return hipSuccess;
    }

    // to[i] = the caller's triple i, wrapped into the box; complete when it returns
    hipError_t upload(const double* from, double4* to, size_t n, const Box& box, hipStream_t stream)
    {
        const size_t per = half_ / (3 * sizeof(double));
        const size_t chunks = (n + per - 1) / per;
        for(size_t c = 0; c < chunks; ++c)
        {
            if(c >= 2)
            {
                const hipError_t e = hipEventSynchronize(ev_[c & 1]);
                if(e != hipSuccess) {return e;}
            }
            const size_t k = std::min(per, n - c * per);
            double* half = reinterpret_cast<double*>(static_cast<char*>(pin_) + (c & 1) * half_);
            std::memcpy(half, from + 3 * c * per, 3 * k * sizeof(double));
            hipLaunchKernelGGL(k_unpack_xyz, dim3((uint32_t)((k + 255) / 256)), dim3(256), 0, stream, half,
                               (uint32_t)(c * per), (uint32_t)k, box, to);
            hipError_t e = hipGetLastError();
            if(e == hipSuccess && chunks > 2) {e = hipEventRecord(ev_[c & 1], stream);}
            if(e != hipSuccess) {return e;}
        }
        return hipStreamSynchronize(stream);
    }

  private:
    void* pin_ = nullptr;
    size_t half_ = 0;
    hipEvent_t ev_[2] = {nullptr, nullptr};
};

} // mjg
