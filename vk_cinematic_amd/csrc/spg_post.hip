// gfx950 kernels for the step after the path: progressive accumulation of
// images across trace calls and the viewer's tone mapping.
#include "spg_internal.h"
#include "spg_tx.h"

namespace spg {

// dst = (dst * before + src * added) / (before + added), RGB; alpha 1.
__global__ __launch_bounds__(256) void k_accumulate(float4 *__restrict__ dst,
                                                    const float4 *__restrict__ src,
                                                    uint32_t pixels, float before,
                                                    float added, float total)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < pixels;
         i = stride_next(i, gridDim.x * 256, pixels))
    {
        float4 a = dst[i], b = src[i];
        a.x = (a.x * before + b.x * added) / total;
        a.y = (a.y * before + b.y * added) / total;
        a.z = (a.z * before + b.z * added) / total;
        a.w = 1.0f;
        dst[i] = a;
    }
}

// The gamma step's byte as a step function of x = c / (1 + c): entry k holds
// the bits of the smallest float x in [0, 1] whose rint(255 g), g the float
// nearest x^(1/2.2f) (the double power rounded once), is at least k.  The
// power is strictly increasing from float to float (neighbours differ by 2.7e-8
// relative, its double evaluation errs by 2^-52), so byte >= k exactly where x
// >= entry k; at the 255 steps the power stays 1.2e-10 relative away from the
// rounding boundary that decides, far more than that error.
static __device__ const uint32_t kToneSteps[256] = {
    0x00000000, 0x35944E0C, 0x374FD767, 0x381FDC21, 0x38A79168, 0x3911A3B3, 0x39627823,
    0x39A3870B, 0x39E00900, 0x3A13870E, 0x3A3C6D56, 0x3A6AD679, 0x3A8F6F7D, 0x3AAC50AF,
    0x3ACC1B21, 0x3AEEDA6C, 0x3B0A4CB8, 0x3B1EB144, 0x3B349FB6, 0x3B4C1CC5, 0x3B652CD9,
    0x3B7FD443, 0x3B8E0B88, 0x3B9CFC9E, 0x3BACBF42, 0x3BBD5551, 0x3BCEC087, 0x3BE102A5,
    0x3BF41D49, 0x3C04090D, 0x3C0E714E, 0x3C194831, 0x3C248E6E, 0x3C3044C4, 0x3C3C6BDC,
    0x3C490473, 0x3C560F27, 0x3C638CAC, 0x3C717D99, 0x3C7FE29D, 0x3C875E23, 0x3C8F059D,
    0x3C96E802, 0x3C9F05A2, 0x3CA75EBE, 0x3CAFF3A6, 0x3CB8C496, 0x3CC1D1DC, 0x3CCB1BB2,
    0x3CD4A264, 0x3CDE6628, 0x3CE86749, 0x3CF2A5FC, 0x3CFD2289, 0x3D03EE91, 0x3D096B07,
    0x3D0F06BF, 0x3D14C1DB, 0x3D1A9C73, 0x3D2096A8, 0x3D26B092, 0x3D2CEA50, 0x3D3343F9,
    0x3D39BDAD, 0x3D405781, 0x3D471197, 0x3D4DEBFD, 0x3D54E6DA, 0x3D5C0239, 0x3D633E42,
    0x3D6A9AFE, 0x3D721896, 0x3D79B711, 0x3D80BB4C, 0x3D84AB98, 0x3D88AC81, 0x3D8CBE0B,
    0x3D90E049, 0x3D95133D, 0x3D9956FC, 0x3D9DAB88, 0x3DA210F5, 0x3DA68744, 0x3DAB0E89,
    0x3DAFA6C6, 0x3DB4500E, 0x3DB90A63, 0x3DBDD5D8, 0x3DC2B26E, 0x3DC7A038, 0x3DCC9F37,
    0x3DD1AF7F, 0x3DD6D110, 0x3DDC03FC, 0x3DE14844, 0x3DE69DFD, 0x3DEC0523, 0x3DF17DCD,
    0x3DF707F8, 0x3DFCA3B8, 0x3E012886, 0x3E040804, 0x3E06F055, 0x3E09E183, 0x3E0CDB8C,
    0x3E0FDE7B, 0x3E12EA4F, 0x3E15FF12, 0x3E191CC1, 0x3E1C4368, 0x3E1F7305, 0x3E22ABA1,
    0x3E25ED3B, 0x3E2937DE, 0x3E2C8B86, 0x3E2FE83F, 0x3E334E07, 0x3E36BCE7, 0x3E3A34DD,
    0x3E3DB5F4, 0x3E414029, 0x3E44D387, 0x3E48700B, 0x3E4C15BF, 0x3E4FC4A1, 0x3E537CBB,
    0x3E573E0A, 0x3E5B089A, 0x3E5EDC66, 0x3E62B97A, 0x3E669FCF, 0x3E6A8F78, 0x3E6E8867,
    0x3E728AB1, 0x3E769649, 0x3E7AAB44, 0x3E7EC993, 0x3E8178A6, 0x3E839130, 0x3E85AE73,
    0x3E87D067, 0x3E89F717, 0x3E8C227B, 0x3E8E529F, 0x3E90877C, 0x3E92C11B, 0x3E94FF75,
    0x3E974296, 0x3E998A75, 0x3E9BD71F, 0x3E9E288A, 0x3EA07EC2, 0x3EA2D9BF, 0x3EA5398D,
    0x3EA79E23, 0x3EAA078D, 0x3EAC75C2, 0x3EAEE8CF, 0x3EB160A9, 0x3EB3DD5E, 0x3EB65EE5,
    0x3EB8E549, 0x3EBB7082, 0x3EBE009B, 0x3EC0958C, 0x3EC32F60, 0x3EC5CE10, 0x3EC871A6,
    0x3ECB1A19, 0x3ECDC777, 0x3ED079B5, 0x3ED330E0, 0x3ED5ECEE, 0x3ED8ADED, 0x3EDB73D1,
    0x3EDE3EA9, 0x3EE10E6A, 0x3EE3E320, 0x3EE6BCC3, 0x3EE99B5E, 0x3EEC7EE8, 0x3EEF676E,
    0x3EF254E5, 0x3EF5475B, 0x3EF83EC5, 0x3EFB3B31, 0x3EFE3C94, 0x3F00A17E, 0x3F02272E,
    0x3F03AF62, 0x3F053A14, 0x3F06C74B, 0x3F085701, 0x3F09E93E, 0x3F0B7DFB, 0x3F0D1540,
    0x3F0EAF08, 0x3F104B58, 0x3F11EA2C, 0x3F138B8A, 0x3F152F6D, 0x3F16D5DC, 0x3F187ED0,
    0x3F1A2A52, 0x3F1BD85A, 0x3F1D88F2, 0x3F1F3C11, 0x3F20F1C1, 0x3F22A9F9, 0x3F2464C3,
    0x3F262218, 0x3F27E1FF, 0x3F29A473, 0x3F2B697A, 0x3F2D310E, 0x3F2EFB37, 0x3F30C7EE,
    0x3F32973C, 0x3F346919, 0x3F363D8E, 0x3F381493, 0x3F39EE31, 0x3F3BCA61, 0x3F3DA92B,
    0x3F3F8A89, 0x3F416E81, 0x3F43550E, 0x3F453E37, 0x3F4729F5, 0x3F491851, 0x3F4B0943,
    0x3F4CFCD5, 0x3F4EF2FE, 0x3F50EBC7, 0x3F52E728, 0x3F54E52B, 0x3F56E5C8, 0x3F58E907,
    0x3F5AEEE1, 0x3F5CF75F, 0x3F5F0279, 0x3F611037, 0x3F632093, 0x3F653394, 0x3F674934,
    0x3F69617B, 0x3F6B7C61, 0x3F6D99EF, 0x3F6FBA1D, 0x3F71DCF5, 0x3F74026F, 0x3F762A92,
    0x3F785558, 0x3F7A82CA, 0x3F7CB2DF, 0x3F7EE5A4};

// PerformToneMapping (src/shaders/post_processing.frag.glsl:19-26):
// c *= exposure; c = c / (1 + c); c = pow(c, 1/2.2); then the UNORM8 write
// of the swapchain: round to nearest of 255 c.  Alpha 255.
//
// kDouble: the bytes of the double-precision power without evaluating it: a
// single-precision estimate of 255 g is off by far less than a step (log2 and
// exp2 to 1e-6), so the byte is its rounding or a neighbour, and two entries of
// the step table (in LDS) decide.  1920x1080: 43 -> 9.9 us (41 MB, 4.2 TB/s;
// the power was ~200 double operations per channel).  8 blocks per CU, each
// loading its table once.
template <bool kDouble>
__global__ __launch_bounds__(256) void k_tonemap(const float4 *__restrict__ src,
                                                 uint32_t pixels, float exposure,
                                                 uchar4 *__restrict__ out)
{
    __shared__ float steps[257];
    if (kDouble)
    {
        steps[threadIdx.x] = __uint_as_float(kToneSteps[threadIdx.x]);
        if (threadIdx.x == 0) steps[256] = INFINITY;
        __syncthreads();
    }
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < pixels;
         i = stride_next(i, gridDim.x * 256, pixels))
    {
        const float4 c = src[i];
        const float ch[3] = {c.x, c.y, c.z};
        uint8_t q[3];
        for (int k = 0; k < 3; ++k)
        {
            float x = ch[k] * exposure;
            x = x / (1.0f + x);
            // NaN and negative inputs give 0 (pow is NaN there, but
            // +infinity, thus 255, at -infinity); above 1: 255
            if (kDouble)
            {
                const bool unit = x >= 0.0f && x <= 1.0f;
                const float g =
                    __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(x) * (1.0f / 2.2f));
                const int e = unit ? min((int)rintf(g * 255.0f), 255) : 0;
                const int at = e - (x < steps[e] ? 1 : 0) + (x >= steps[e + 1] ? 1 : 0);
                q[k] = (uint8_t)(unit ? at : x > 1.0f || x == -INFINITY ? 255 : 0);
            }
            else
            {
                float g = __powf(x, 1.0f / 2.2f);
                g = clamp_sel(g, 0.0f, 1.0f);
                q[k] = (uint8_t)(uint32_t)rintf(g * 255.0f);
            }
        }
        out[i] = make_uchar4(q[0], q[1], q[2], 255);
    }
}

hipError_t launch_accumulate(hipStream_t s, float4 *dst, const float4 *src,
                             uint32_t pixels, uint32_t before, uint32_t added)
{
    if (pixels == 0) return hipSuccess;
    const uint32_t blocks = stride_blocks(pixels, 256, 65535u);
    k_accumulate<<<blocks, 256, 0, s>>>(dst, src, pixels, (float)before, (float)added,
                                        (float)before + (float)added);
    return hipGetLastError();
}

hipError_t launch_tonemap(hipStream_t s, const float4 *src, uint32_t pixels,
                          float exposure, bool dbl, uchar4 *out)
{
    if (pixels == 0) return hipSuccess;
    const uint32_t most = dbl ? 2048u : 65535u;
    const uint32_t grid = stride_blocks(pixels, 256, most);
    if (dbl) k_tonemap<true><<<grid, 256, 0, s>>>(src, pixels, exposure, out);
    else k_tonemap<false><<<grid, 256, 0, s>>>(src, pixels, exposure, out);
    return hipGetLastError();
}

}  // namespace spg
