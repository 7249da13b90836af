// Stereo matching of a rectified left/right pair for gfx950
// (Frame::ComputeStereoMatch, src/Frame.cpp:150-328):
//   k_stereo        one wave per left keypoint: row-band + octave +
//                   disparity gating of the right keypoints in index order,
//                   top-2 Hamming, ratio 0.70 / threshold 34, 11x11 SAD over
//                   11 shifts on the pyramid level, parabola sub-pixel fit
//   k_stereo_median one workgroup per pair: the median of the accepted SADs,
//                   those beyond 1.6x / below 0.4x of it dropped
// Included by mcv_api.hip (uses LevelDesc, wave_sum).
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcv {

struct StereoJob {
    const float* kl;        // left keypoints (mcv_keypoint rows of 6 x 4 B)
    const uint8_t* dl;
    const int* nl;          // device count
    const float* kr;
    const uint8_t* dr;
    const int* nr;
    int lvl_l, lvl_r;       // LevelDesc index of level 0 of the left / right image
    float* u_right;         // per left keypoint, -1 when unmatched
    float* depth;
    int* sad;               // per left keypoint, -1 when unmatched
};

struct StereoParams {
    float scale[16], inv_scale[16];
    float bf, b;
    int cap;
};

__global__ __launch_bounds__(256) void k_stereo(const StereoJob* jobs, const LevelDesc* lv, const uint8_t* pyr,
                                                StereoParams sp) {
    const StereoJob J = jobs[blockIdx.y];
    const int iL = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int nl = min(*J.nl, sp.cap), nr = min(*J.nr, sp.cap);
    if (iL >= nl) return;
    const float* kp = J.kl + 6 * iL;
    const float uL = kp[0], vL = kp[1];
    const int levelL = reinterpret_cast<const int*>(kp)[5];
    bool ok = true;
    if (lane == 0) {
        J.u_right[iL] = -1.f;
        J.depth[iL] = -1.f;
        J.sad[iL] = -1;
    }
    const int rowL = (int)vL;
    const float minZ = sp.b, minD = 1.f;
    const float maxD = fminf(sp.bf / minZ, 1000.0f);
    const float minU = uL - maxD, maxU = uL - minD;
    if (maxU < 0) return;
    uint32_t q[8];
    const uint32_t* qd = reinterpret_cast<const uint32_t*>(J.dl + 32ll * iL);
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = qd[k];
    uint32_t k0 = 999u << 22, k1 = 999u << 22;
    int ncand = 0;
    // 4 right keypoints per lane in flight (2000 against 2000 keypoints 21 us; 24
    // when the scan waited for each)
    for (int r0 = lane; r0 < nr; r0 += 256) {
        float kx[4], ky[4];
        int ko[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float* kr = J.kr + 6 * min(r0 + 64 * u, nr - 1);
            kx[u] = kr[0];
            ky[u] = kr[1];
            ko[u] = reinterpret_cast<const int*>(kr)[5];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int iR = r0 + 64 * u;
            if (iR >= nr) break;
            const float kpY = ky[u];
            const int oR = ko[u];
            const float r = 10.f * sp.scale[oR];
            const int maxr = (int)ceilf(kpY + r), minr = (int)floorf(kpY - r);
            if (rowL < minr || rowL > maxr) continue;
            if (oR < levelL - 1 || oR > levelL + 1) continue;
            const float uR = kx[u];
            if (!(uR >= minU && uR <= maxU)) continue;
            const uint32_t* td = reinterpret_cast<const uint32_t*>(J.dr + 32ll * iR);
            uint32_t d = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) d += __builtin_popcount(q[k] ^ td[k]);
            const uint32_t key = (d << 22) | (uint32_t)iR;
            k1 = min(k1, max(k0, key));
            k0 = min(k0, key);
            ncand++;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t b0 = __shfl_xor(k0, off, 64), b1 = __shfl_xor(k1, off, 64);
        const uint32_t n1 = min(max(k0, b0), min(k1, b1));
        k0 = min(k0, b0);
        k1 = n1;
        ncand += __shfl_xor(ncand, off, 64);
    }
    const float d0 = (float)(k0 >> 22), d1 = (float)(k1 >> 22);
    if (ncand == 0 || !(d0 / d1 <= 0.70f) || d0 > (float)34) ok = false;
    if (!ok) return;
    const int iR = (int)(k0 & ((1u << 22) - 1));
    const float uR0 = J.kr[6 * iR];
    const float scaleFactor = sp.inv_scale[levelL];
    const float scaleduL = roundf(uL * scaleFactor);
    const float scaledvL = roundf(vL * scaleFactor);
    const float scaleduR0 = roundf(uR0 * scaleFactor);
    const int w = 5, L = 5;
    const LevelDesc DL = lv[J.lvl_l + levelL], DR = lv[J.lvl_r + levelL];
    if (scaledvL - w < 0 || scaledvL + w + 1 >= DL.h || scaleduL - w < 0 || scaleduL + w + 1 >= DL.w) return;
    const float iniu = scaleduR0 + L - w, endu = scaleduR0 + L + w + 1;
    if (iniu < 0 || endu >= DR.w) return;
    if (scaleduR0 - L - w < 0) return;  // the reference's colRange would assert
    const uint8_t* IL = pyr + DL.pix;
    const uint8_t* IR = pyr + DR.pix;
    const int y0 = (int)scaledvL - w, xl = (int)scaleduL - w;
    const int cl = IL[(long long)(y0 + w) * DL.pitch + xl + w];
    int bestDist = 0x7FFFFFFF, bestincR = 0;
    float vd[2 * 5 + 1];
#pragma unroll
    for (int incR = -L; incR <= L; incR++) {
        const int xr = (int)scaleduR0 + incR - w;
        const int cr = IR[(long long)(y0 + w) * DR.pitch + xr + w];
        int acc = 0;
        for (int p = lane; p < 121; p += 64) {
            const int yy = p / 11, xx = p - 11 * yy;
            const int a = (int)IL[(long long)(y0 + yy) * DL.pitch + xl + xx] - cl;
            const int b = (int)IR[(long long)(y0 + yy) * DR.pitch + xr + xx] - cr;
            acc += abs(a - b);
        }
        acc = wave_sum(acc);
        const float dist = (float)acc;
        if (dist < (float)bestDist) {
            bestDist = (int)dist;
            bestincR = incR;
        }
        vd[L + incR] = dist;
    }
    if (lane != 0) return;
    if (bestincR == -L || bestincR == L) return;
    float dist1 = 0, dist2 = 0, dist3 = 0;
#pragma unroll
    for (int k = 1; k < 2 * L; k++)
        if (k == L + bestincR) {
            dist1 = vd[k - 1];
            dist2 = vd[k];
            dist3 = vd[k + 1];
        }
    const float deltaR = (dist1 - dist3) / (2.0f * (dist1 + dist3 - 2.0f * dist2));
    if (deltaR < -1 || deltaR > 1) return;
    const float bestuR = sp.scale[levelL] * ((float)scaleduR0 + (float)bestincR + deltaR);
    const float disparity = uL - bestuR;
    if (disparity >= minD && disparity < maxD) {
        J.depth[iL] = sp.bf / disparity;
        J.u_right[iL] = bestuR;
        J.sad[iL] = bestDist;
    }
}

constexpr int kStereoMedianCap = 8192;

// The reference sorts the accepted (SAD, index) pairs and drops entries from
// the end while the SAD exceeds 1.6 times that of the middle entry (n / 2) and
// from the start while it is below 0.4 times: SADs of the middle one's size
// always stay, so both are a test of each entry alone and only the middle SAD
// is needed.  A SAD is below 2^16 (121 pixels of at most 510), so two counts
// of 256 bins find it; the SADs stay in registers.  Latency bound: one
// workgroup per pair (sorting 2000 pairs took 52 us).
__global__ __launch_bounds__(1024) void k_stereo_median(const StereoJob* jobs, StereoParams sp) {
    constexpr int kPer = kStereoMedianCap / 1024;
    __shared__ int s_bin[2][256];
    __shared__ int s_sel[2], s_rank[2];
    const StereoJob J = jobs[blockIdx.x];
    const int nl = min(min(*J.nl, sp.cap), kStereoMedianCap);
    int sad[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int i = u * 1024 + threadIdx.x;
        sad[u] = i < nl ? J.sad[i] : -1;
    }
    if (threadIdx.x < 512) s_bin[0][threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll
        for (int u = 0; u < kPer; u++)
            if (sad[u] >= 0 && (pass == 0 || (sad[u] >> 8) == s_sel[0]))
                atomicAdd(&s_bin[pass][pass == 0 ? sad[u] >> 8 : sad[u] & 255], 1);
        __syncthreads();
        if (threadIdx.x < 64) {
            // lane l: bins 4 l .. 4 l + 3
            const int l = threadIdx.x;
            int c[4], sum = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                c[k] = s_bin[pass][4 * l + k];
                sum += c[k];
            }
            int incl = sum;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if (l >= o) incl += y;
            }
            const int rank = pass == 0 ? __shfl(incl, 63, 64) / 2 : s_rank[0];
            // the bin that holds the rank-th entry (no lane when there is none)
            int before = incl - sum;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (rank >= before && rank < before + c[k]) {
                    s_sel[pass] = 4 * l + k;
                    s_rank[pass] = rank - before;
                }
                before += c[k];
            }
            if (pass == 0 && l == 63 && incl == 0) s_sel[0] = -1;
        }
        __syncthreads();
        if (s_sel[0] < 0) return;  // nothing accepted
    }
    const float median = (float)(s_sel[0] << 8 | s_sel[1]);
    const float th_max = 1.6f * median;
    const float th_min = (float)(0.4 * (double)median);
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int i = u * 1024 + threadIdx.x;
        if (sad[u] >= 0 && ((float)sad[u] > th_max || (float)sad[u] < th_min)) {
            J.u_right[i] = -1.f;
            J.depth[i] = -1.f;
            J.sad[i] = -1;
        }
    }
}

}  // namespace mcv
