// Generated by gen_math_constants.py -- do not edit by hand.
// Each value is the correctly rounded binary64/binary32 image of an exact
// mathematical constant computed with 100-digit decimal arithmetic, except
// the minimax tables SIN64, COS64, EXP64, ATAN64 and ATAN01_MM32 (Remez
// exchanges).
#pragma once

namespace u1m {
static constexpr double K_PI = 0x1.921fb54442d18p+1;  // 3.141592653589793
static constexpr double K_TWO_PI = 0x1.921fb54442d18p+2;  // 6.283185307179586
static constexpr double K_PI_LO = 0x1.1a62633145c07p-53;  // 1.2246467991473532e-16
static constexpr double K_TWO_PI_LO = 0x1.1a62633145c07p-52;  // 2.4492935982947064e-16
static constexpr double K_PIO2_HI = 0x1.921fb54442d18p+0;  // 1.5707963267948966
static constexpr double K_PIO2_LO = 0x1.1a62633145c07p-54;  // 6.123233995736766e-17
static constexpr double K_PIO4 = 0x1.921fb54442d18p-1;  // 0.7853981633974483
static constexpr double K_PIO4_LO = 0x1.1a62633145c07p-55;  // 3.061616997868383e-17
static constexpr double K_TWO_OVER_PI = 0x1.45f306dc9c883p-1;  // 0.6366197723675814
static constexpr double K_PIO2_1 = 0x1.921fb54442d18p+0;  // 1.5707963267948966
static constexpr double K_PIO2_2 = 0x1.1a62633145c07p-54;  // 6.123233995736766e-17
static constexpr double K_PIO2_3 = -0x1.f1976b7ed8fbcp-110;  // -1.4973849048591698e-33
static constexpr double K_LN2_HI = 0x1.62e42fefa39efp-1;  // 0.6931471805599453
static constexpr double K_LN2_LO = 0x1.abc9e3b39803fp-56;  // 2.3190468138462996e-17
static constexpr double K_LOG2E = 0x1.71547652b82fep+0;  // 1.4426950408889634
static constexpr double K_TAN_PIO8 = 0x1.a827999fcef32p-2;  // 0.41421356237309503
static constexpr float KF_PI = 0x1.921fb60000000p+1f;  // 3.1415927410125732
static constexpr float KF_TWO_PI = 0x1.921fb60000000p+2f;  // 6.2831854820251465
static constexpr float KF_PIO2_HI = 0x1.921fb60000000p+0f;  // 1.5707963705062866
static constexpr float KF_PIO2_LO = -0x1.777a5c0000000p-25f;  // -4.371138828673793e-08
static constexpr float KF_PIO4 = 0x1.921fb60000000p-1f;  // 0.7853981852531433
static constexpr float KF_TWO_OVER_PI = 0x1.45f3060000000p-1f;  // 0.6366197466850281
static constexpr float KF_PIO2_1 = 0x1.921fb60000000p+0f;  // 1.5707963705062866
static constexpr float KF_PIO2_2 = -0x1.777a5c0000000p-25f;  // -4.371138828673793e-08
static constexpr float KF_PIO2_3 = -0x1.ee59da0000000p-50f;  // -1.7151245100058819e-15
static constexpr float KF_TAN_PIO8 = 0x1.a8279a0000000p-2f;  // 0.4142135679721832
static constexpr int N_SIN64 = 6;
#define U1M_SIN64_COEFFS 0x1.5d8ff90144cdcp-33, -0x1.ae5e5b1533e8ep-26, 0x1.71de356876082p-19, -0x1.a01a019bfea3dp-13, 0x1.111111110f7d6p-7, -0x1.5555555555548p-3
static constexpr int N_COS64 = 7;
#define U1M_COS64_COEFFS -0x1.8f7571988e6d6p-37, 0x1.1ee96d22197a9p-29, -0x1.27e4f72c0286ep-22, 0x1.a01a019b2e602p-16, -0x1.6c16c16c13bb1p-10, 0x1.5555555555539p-5, -0x1.0000000000000p-1
static constexpr int N_EXP64 = 11;
#define U1M_EXP64_COEFFS 0x1.1e3d557e25f52p-29, 0x1.af6bad920703bp-26, 0x1.27e5b3f37a4fbp-22, 0x1.71ddf0419bf66p-19, 0x1.a01a0136d60b9p-16, 0x1.a01a01b3715f4p-13, 0x1.6c16c16c30321p-10, 0x1.111111110ec7ep-7, 0x1.5555555555503p-5, 0x1.555555555555bp-3, 0x1.0000000000000p-1
static constexpr int N_ATAN64 = 11;
#define U1M_ATAN64_COEFFS -0x1.2565a607b5743p-6, 0x1.37d2c7d80af0ap-5, -0x1.9cd14a1039218p-5, 0x1.df0ee3b60d900p-5, -0x1.10ebaf736a466p-4, 0x1.3b11182728061p-4, -0x1.745cf8cb68c93p-4, 0x1.c71c70e552a3ap-4, -0x1.24924922aaf63p-3, 0x1.99999999957e7p-3, -0x1.555555555553dp-2
static constexpr int N_BESI0_64 = 27;
#define U1M_BESI0_64_COEFFS 0x1.2d843c1f0a6f9p-177, 0x1.8e189760fbc74p-168, 0x1.e5f504c9e358cp-159, 0x1.1159d2b18fe1fp-149, 0x1.1a6d4e307528fp-140, 0x1.0afb53e9cec0bp-131, 0x1.cbeaf38dc529fp-123, 0x1.674f8e46c208cp-114, 0x1.faaf2fa1c79e5p-106, 0x1.40a2dc2460523p-97, 0x1.69f7da8510bcdp-89, 0x1.69f7da8510bcdp-81, 0x1.3e22d70ef3b5fp-73, 0x1.e725594ee52e9p-66, 0x1.4197a7f5154bcp-58, 0x1.69ca9cf3b7f54p-51, 0x1.5601885e63e5dp-44, 0x1.0b313289be0b9p-37, 0x1.522a43f65486ap-31, 0x1.522a43f65486ap-25, 0x1.02e85c0898b71p-19, 0x1.23456789abcdfp-14, 0x1.c71c71c71c71cp-10, 0x1.c71c71c71c71cp-6, 0x1.0000000000000p-2, 0x1.0000000000000p+0, 0x1.0000000000000p+0
static constexpr int N_BESI1_64 = 27;
#define U1M_BESI1_64_COEFFS 0x1.655a5a37c0843p-182, 0x1.e9f6e1b270f54p-173, 0x1.37033643c4b3bp-163, 0x1.6c77c3976a829p-154, 0x1.88f11edf3ed4cp-145, 0x1.84564b82a1184p-136, 0x1.5e69de22df5cep-127, 0x1.1f72d8389b3a3p-118, 0x1.aaae78f4066a6p-110, 0x1.1d028acb00491p-101, 0x1.54ad09e6a6575p-93, 0x1.69f7da8510bcdp-85, 0x1.53585cdcbfb10p-77, 0x1.165e7c2d153f3p-69, 0x1.8bce58901a35ep-62, 0x1.e2637bef9ff1ap-55, 0x1.f17697cf1cf13p-48, 0x1.ab81ea75fcdf4p-41, 0x1.2c9758daf5cd0p-34, 0x1.522a43f65486ap-28, 0x1.27e4fb7789f5cp-22, 0x1.845c8a0ce5129p-17, 0x1.6c16c16c16c17p-12, 0x1.c71c71c71c71cp-8, 0x1.5555555555555p-4, 0x1.0000000000000p-1, 0x1.0000000000000p+0
static constexpr int N_SIN32 = 4;
#define U1M_SIN32_COEFFS 0x1.71de3a0000000p-19f, -0x1.a01a020000000p-13f, 0x1.1111120000000p-7f, -0x1.5555560000000p-3f
static constexpr int N_COS32 = 5;
#define U1M_COS32_COEFFS -0x1.27e4fc0000000p-22f, 0x1.a01a020000000p-16f, -0x1.6c16c20000000p-10f, 0x1.5555560000000p-5f, -0x1.0000000000000p-1f
static constexpr int N_ATAN32 = 9;
#define U1M_ATAN32_COEFFS -0x1.af286c0000000p-5f, 0x1.e1e1e20000000p-5f, -0x1.1111120000000p-4f, 0x1.3b13b20000000p-4f, -0x1.745d180000000p-4f, 0x1.c71c720000000p-4f, -0x1.24924a0000000p-3f, 0x1.99999a0000000p-3f, -0x1.5555560000000p-2f
static constexpr int N_ATAN01_MM32 = 8;
#define U1M_ATAN01_MM32_COEFFS 0x1.7ed2320000000p-9f, -0x1.0c2c140000000p-6f, 0x1.61fdda0000000p-5f, -0x1.3556b60000000p-4f, 0x1.b4e12a0000000p-4f, -0x1.230adc0000000p-3f, 0x1.9978f40000000p-3f, -0x1.5554dc0000000p-2f
}  // namespace u1m
