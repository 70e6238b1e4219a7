// dst_f64.hip -- the FP64 DST passes at every transform length the plans accept
// (M = 2 n, n = 2..1024 with factors 2, 3, 5), in eight parts that the build
// compiles side by side (IBPM_DST_PART), split for equal compile time.
#include "dst_passes.h"

#if IBPM_DST_PART == 0
#define IBPM_LENGTHS(X) X(4) X(48) X(96) X(180) X(288) X(432) X(576) X(768) X(960) X(1200) X(1600)
#elif IBPM_DST_PART == 1
#define IBPM_LENGTHS(X) X(6) X(50) X(100) X(192) X(300) X(450) X(600) X(800) X(972) X(1250) X(1620)
#elif IBPM_DST_PART == 2
#define IBPM_LENGTHS(X) X(8) X(54) X(108) X(200) X(320) X(480) X(640) X(810) X(1000) X(1280) X(1728)
#elif IBPM_DST_PART == 3
#define IBPM_LENGTHS(X) X(10) X(60) X(120) X(216) X(324) X(486) X(648) X(864) X(1024) X(1296) X(1800)
#elif IBPM_DST_PART == 4
#define IBPM_LENGTHS(X) X(12) X(64) X(128) X(240) X(360) X(500) X(720) X(900) X(1080) X(1350) X(1920)
#elif IBPM_DST_PART == 5
#define IBPM_LENGTHS(X) X(16) X(18) X(72) X(144) X(250) X(384) X(512) X(750) X(1152) X(1440) X(1944)
#elif IBPM_DST_PART == 6
#define IBPM_LENGTHS(X) X(20) X(24) X(80) X(150) X(256) X(400) X(540) X(1458) X(1500) X(2000)
#else
#define IBPM_LENGTHS(X) X(30) X(32) X(36) X(40) X(90) X(160) X(162) X(270) X(1536) X(2048)
#endif

namespace ibpmg {

#define IBPM_DST_NAME2(k) launch_dst_##k
#define IBPM_DST_NAME(k) IBPM_DST_NAME2(k)
#define IBPM_CASE(M)                         \
    case M:                                  \
        if (L.njobs) launch_dst_len<M>(L);   \
        return true;

bool IBPM_DST_NAME(IBPM_DST_PART)(const DstLaunch& L) {
    switch (L.M) {
        IBPM_LENGTHS(IBPM_CASE)
    default: return false;
    }
}

}  // namespace ibpmg
