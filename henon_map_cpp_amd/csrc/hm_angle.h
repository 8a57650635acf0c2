// atan2 for the Birkhoff sums, by a table in LDS: with ax = |x|, ay = |y|, mx and mn the
// larger and the smaller, i the nearest integer to 64 mn / mx and c = i / 64,
//   atan(mn / mx) = atan(c) + atan(u),  u = (mn - c mx) / (mx + c mn),  |u| <= 1/127,
// atan(u) by four terms of its series (the fifth is below 2e-18 u). The table holds the
// octant's angle at c in two parts, so what atan(u) joins is exact to 2^-106 and the last
// sum is the only rounding to count where i > 0 or the octant is not the first: a mean
// error of 0.37 units of 2^-53 of the result, that of a correctly rounded atan2 and of a
// good library's (0.51 with the octant taken apart from a rounded table entry), at most
// 3.0 found, in the first octant near the axis. Signs as the library's, those of zeros included.
// Sums of magnitudes outside [2^-500, 2^500] (zero, subnormal, huge, infinite) are brought
// into range first, on a branch of the whole wavefront; NaN passes through (the lost lanes
// of a wavefront hold it, turn after turn). About 45 instructions and three constants,
// where the library's takes about 65 and twenty, which the compiler keeps in registers
// through a loop.
// Compiles as host code too (no HIP types), so a host check can build it alone.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#define HM_ANGLE_FN __host__ __device__ inline
#else
#define HM_ANGLE_FN inline
#endif

namespace hm {

constexpr int kAngleBins = 65;
struct alignas(16) AngleEntry {
    double hi, lo;  // the angle, rounded, and what is left of it
};
constexpr int kAngleEntries = 4 * kAngleBins;

// With a = atan(i / 64), i = 0 .. 64: a, pi/2 - a, pi - a, pi/2 + a.
#if defined(__HIPCC__)
__device__
#endif
static const AngleEntry kAtan[kAngleEntries] = {
    {0.0, 0.0}, {0x1.921fb54442d18p0, 0x1.1a62633145c07p-54}, {0x1.921fb54442d18p1, 0x1.1a62633145c07p-53},
    {0x1.921fb54442d18p0, 0x1.1a62633145c07p-54}, {0x1.fff555bbb729bp-7, -0x1.220c39d4dff50p-61},
    {0x1.8e1fca98cb633p0, 0x1.1299ee93be016p-56}, {0x1.901fbfee871a6p1, -0x1.507b9094e55fap-53},
    {0x1.961f9fefba3fdp0, 0x1.f01e4abd9c008p-54}, {0x1.ffd55bba97625p-6, -0x1.5ec431444912cp-60},
    {0x1.8a205fd558740p0, -0x1.30228c09a91b4p-54}, {0x1.8e200a8ccda2cp1, -0x1.5c028d8635ad9p-58},
    {0x1.9a1f0ab32d2f1p0, -0x1.36315b2796c7cp-55}, {0x1.7fb818430da2ap-5, -0x1.86ef8f794f105p-63},
    {0x1.8621f4822a647p0, -0x1.26d12837ecc05p-57}, {0x1.8c20d4e3369b0p1, -0x1.853be0eadbebdp-53},
    {0x1.9e1d76065b3eap0, -0x1.a661149676e72p-54}, {0x1.ff55bb72cfdeap-5, -0x1.c934d86d23f1dp-60},
    {0x1.82250768ac529p0, -0x1.e78c96d05afcbp-58}, {0x1.8a225e5677921p1, -0x1.820b331ddff7bp-53},
    {0x1.a21a631fd9508p0, -0x1.acc270306ecf6p-54}, {0x1.3f59f0e7c559dp-4, 0x1.ac4ce285df847p-58},
    {0x1.7e2a1635c67bep0, 0x1.bf9d9508e7c82p-54}, {0x1.8824e5bd04a6bp1, 0x1.6cfffc1d16c45p-53},
    {0x1.a6155452bf272p0, 0x1.d49cc5668ee2dp-56}, {0x1.7ee182602f10fp-4, -0x1.cfb654c0c3d98p-58},
    {0x1.7a319d1e3fe07p0, 0x1.775dc87d51fe0p-54}, {0x1.8628a93141590p1, -0x1.6e3fd45168419p-54},
    {0x1.aa0dcd6a45c29p0, 0x1.7acdfbca7305bp-55}, {0x1.be39ebe6f07c3p-4, 0x1.f7b8f29a05987p-58},
    {0x1.763c1685d3c9cp0, 0x1.d736a03d2b373p-57}, {0x1.842de5e50b4dap1, 0x1.55493738eb275p-54},
    {0x1.ae035402b1d94p0, 0x1.f9ddf25ae619fp-54}, {0x1.fd5ba9aac2f6ep-4, -0x1.cd37686760c17p-59},
    {0x1.7249faa996a21p0, 0x1.a8cc1e7480c68p-54}, {0x1.8234d7f6ecb9dp1, -0x1.3cd17e5a39792p-54},
    {0x1.b1f56fdeef00fp0, 0x1.17f14fdc1574cp-55}, {0x1.1e1fafb043727p-3, -0x1.b485914dacf8cp-59},
    {0x1.6e5bbf4e3a633p0, 0x1.a8068fbbb3283p-54}, {0x1.803dba493e9a6p1, -0x1.3d970d1307176p-54},
    {0x1.b5e3ab3a4b3fdp0, 0x1.197c6d4db0b15p-55}, {0x1.3d6eee8c6626cp-3, 0x1.61a3b0ce9281bp-57},
    {0x1.6a71d772b60cbp0, -0x1.11d212e88c8fdp-54}, {0x1.7e48c65b7c6f2p1, -0x1.fbb7d7dba367bp-53},
    {0x1.b9cd9315cf966p0, -0x1.72d24d69cfdebp-55}, {0x1.5c9811e3ec26ap-3, -0x1.054ab2c010f3dp-58},
    {0x1.668cb307c54cbp0, 0x1.55b872ea367d6p-57}, {0x1.7c563426040f2p1, -0x1.5d734738b9b7fp-53},
    {0x1.bdb2b780c0566p0, -0x1.f5f247fabb4edp-54}, {0x1.7b97b4bce5b02p-3, 0x1.347b0b4f881cap-58},
    {0x1.62acbeaca61b8p0, 0x1.c6ac9f134fa91p-60}, {0x1.7a6639f874768p1, 0x1.217d15ad92ff1p-54},
    {0x1.c192abdbdf879p0, -0x1.d255ec19c1bddp-54}, {0x1.9a6a8e96c8626p-3, 0x1.cf601e7b4348ep-59},
    {0x1.5ed2637169c54p0, -0x1.f4189dc29459ep-54}, {0x1.78790c5ad64b6p1, -0x1.b36c75229d32dp-55},
    {0x1.c56d07171bdddp0, 0x1.46eb2128fed5ap-57}, {0x1.b90d7529260a2p-3, 0x1.17b10d2e0e5abp-61},
    {0x1.5afe069f1e104p0, 0x1.8330116e9a3b9p-58}, {0x1.768eddf1b070ep1, 0x1.329564482f642p-54},
    {0x1.c94163e96792dp0, -0x1.e36e3ab45e22ep-54}, {0x1.d77d5df205736p-3, 0x1.c648d1534597ep-57},
    {0x1.5730098602231p0, 0x1.e1994906dd0d7p-54}, {0x1.74a7df65227a5p1, -0x1.040453c7dd322p-54},
    {0x1.cd0f6102837ffp0, 0x1.4cadf56eb9cdap-56}, {0x1.f5b75f92c80ddp-3, 0x1.8ab6e3cf7afbdp-57},
    {0x1.5368c951e9cfdp0, -0x1.96f47948a99f1p-54}, {0x1.72c43f4b1650ap1, 0x1.c1b6f4f44e10bp-53},
    {0x1.d0d6a1369bd34p0, -0x1.a23602a65700cp-57}, {0x1.09dc597d86362p-2, 0x1.62e47390cb865p-56},
    {0x1.4fa89ee4e1440p0, -0x1.3e56b9b2ed212p-54}, {0x1.70e42a14920acp1, -0x1.1fa2b40d3b05dp-57},
    {0x1.d496cba3a45f1p0, -0x1.19c8ffd50ebc0p-55}, {0x1.18bf5a30bf178p-2, 0x1.30ca4748b1bf9p-57},
    {0x1.4befdeb8130bap0, 0x1.e89234905f110p-55}, {0x1.6f07c9fe2aee9p1, 0x1.0755bebcbaa47p-53},
    {0x1.d84f8bd072976p0, 0x1.407bac1a5bf86p-54}, {0x1.278372057ef46p-2, -0x1.077cdd36dfc81p-56},
    {0x1.483ed8c2e3147p0, -0x1.477ccb02049b2p-55}, {0x1.6d2f470392f30p1, -0x1.c4ae0127de469p-53},
    {0x1.dc0091c5a28eap0, -0x1.277cd41c72319p-54}, {0x1.362773707ebccp-2, -0x1.963a544b672d8p-57},
    {0x1.4495d86823225p0, 0x1.4d29adbab2a62p-54}, {0x1.6b5ac6d632f9fp1, -0x1.9873ef1407997p-54},
    {0x1.dfa992206280bp0, 0x1.cf36314fb1b58p-55}, {0x1.44aa436c2af0ap-2, -0x1.5d5e43c55b3bap-56},
    {0x1.40f5246938156p0, -0x1.1c8c17bac6e15p-55}, {0x1.698a6cd6bd737p1, 0x1.1838aea7c49f9p-55},
    {0x1.e34a461f4d8dbp0, -0x1.3cf52dc0110e8p-54}, {0x1.530ad9951cd4ap-2, -0x1.2566480884082p-57},
    {0x1.3d5cfedefb9c6p0, -0x1.81e1a79b537d2p-55}, {0x1.67be5a119f36fp1, 0x1.65c63d8e70078p-56},
    {0x1.e6e26ba98a06bp0, -0x1.0a4a65cfcac09p-54}, {0x1.614840309cfe2p-2, -0x1.a725715711f00p-56},
    {0x1.39cda5381b920p0, -0x1.ef5101e3d70e5p-56}, {0x1.65f6ad3e2f31cp1, 0x1.3d1c45709ff9bp-55},
    {0x1.ea71c5506a111p0, -0x1.4f66f9247ebb9p-54}, {0x1.6f61941e4def1p-2, -0x1.c63aae6f6e918p-56},
    {0x1.3647503caf55cp0, 0x1.17e21d9a42c9ap-55}, {0x1.643382c07913ap1, 0x1.a65371fe67254p-54},
    {0x1.edf81a4bd64d4p0, 0x1.a8d3b7956a1c1p-54}, {0x1.7d5604b63b3f7p-2, 0x1.69c885c2b249ap-56},
    {0x1.32ca3416b401ap0, 0x1.bff041c0992e0p-54}, {0x1.6274f4ad7b699p1, 0x1.6d295278ef774p-53},
    {0x1.f1753671d1a16p0, 0x1.d3521287c94b6p-56}, {0x1.8b24d394a1b25p-2, 0x1.b6d0ba3748fa8p-56},
    {0x1.2f56805f1a64fp0, -0x1.4d472d7231f8dp-56}, {0x1.60bb1ad1ae9b4p1, -0x1.9c77b415a35eep-53},
    {0x1.f4e8ea296b3e2p0, -0x1.77e96e40e800fp-54}, {0x1.98cd5454d6b18p-2, 0x1.9e6c988fd0a77p-56},
    {0x1.2bec602f0d252p0, 0x1.658e7a1aa32d2p-55}, {0x1.5f060ab9a7fb5p1, 0x1.cd29a03e97570p-54},
    {0x1.f8530a59787dep0, 0x1.81fd895539ea5p-54}, {0x1.a64eec3cc23fdp-2, -0x1.24dec1b50b7ffp-56},
    {0x1.288bfa3512419p0, 0x1.8e684e7a2281bp-56}, {0x1.5d55d7bcaa899p1, -0x1.4101c49818cf9p-53},
    {0x1.fbb3705373617p0, 0x1.d12ab2c402e07p-54}, {0x1.b3a911da65c6cp-2, 0x1.ae187b1ca5040p-56},
    {0x1.253570cda95fdp0, 0x1.5db888d438feep-55}, {0x1.5baa9308f618bp1, -0x1.1b60ac324ee01p-53},
    {0x1.ff09f9badc433p0, 0x1.85e881f86f017p-54}, {0x1.c0db4c94ec9f0p-2, -0x1.cc1ce70934c34p-56},
    {0x1.21e8e21f07a9cp0, 0x1.8d699cf392f14p-54}, {0x1.5a044bb1a53dap1, 0x1.53e600126c58dp-53},
    {0x1.012b4434befcap1, 0x1.4eb652ddf11f4p-55}, {0x1.cde53432c1351p-2, -0x1.a2cfa4418f1adp-56},
    {0x1.1ea6683792844p0, 0x1.062c9883530e4p-55}, {0x1.58630ebdeaaaep1, 0x1.9d78af72ef479p-54},
    {0x1.02cc8128798f6p1, 0x1.b1ae7a20e1f9cp-54}, {0x1.dac670561bb4fp-2, 0x1.a2b7f222f65e2p-56},
    {0x1.1b6e192ebbe44p0, 0x1.b1b466a88828ep-54}, {0x1.56c6e7397f5aep1, 0x1.660b64ece6f4bp-53},
    {0x1.0468a8ace4df6p1, 0x1.0620bf7406affp-55}, {0x1.e77eb7f175a34p-2, 0x1.0e53dc1bf3435p-56},
    {0x1.18400747e568bp0, 0x1.ad9ad85491df3p-55}, {0x1.552fde46141d2p1, -0x1.0768185238a80p-53},
    {0x1.05ffb1a0501d3p1, -0x1.510452e3deb76p-53}, {0x1.f40dd0b541418p-2, -0x1.a3992dc382a23p-57},
    {0x1.151c4116f2812p0, 0x1.4ed588e9b614bp-54}, {0x1.539dfb2d9aa95p1, 0x1.349bf60d7dea9p-53},
    {0x1.079194b8c990fp1, 0x1.cbde7af1aad85p-55}, {0x1.0039c73c1a40cp-1, -0x1.b32c949c9d593p-55},
    {0x1.1202d1a635b12p0, 0x1.f3f8ad7f946d1p-54}, {0x1.521143753c415p1, 0x1.872d88586d16cp-53},
    {0x1.091e4c7127f8fp1, 0x1.0330638bdc4f5p-56}, {0x1.0657e94db30d0p-1, -0x1.d5b495f6349e6p-56},
    {0x1.0ef3c09d694b0p0, 0x1.8fcf88aed2e80p-54}, {0x1.5089baf0d60e4p1, 0x1.5518f5f00c544p-53},
    {0x1.0aa5d4f58e2c0p1, 0x1.49ea7b677131bp-55}, {0x1.0c6145b5b43dap-1, 0x1.974fa13b5404fp-58},
    {0x1.0bef126968b2bp0, 0x1.00ed691d90802p-54}, {0x1.4f0763d6d5c22p1, -0x1.e4b033b129bf7p-54},
    {0x1.0c282c0f8e783p1, -0x1.6614515d827fap-53}, {0x1.1255d9bfbd2a9p-1, -0x1.2bdaee1c0ee35p-58},
    {0x1.08f4c864643c4p0, -0x1.a5bfdbd9f2a2cp-55}, {0x1.4d8a3ed45386ep1, 0x1.1e09d51131bc4p-56},
    {0x1.0da5511210b36p1, 0x1.83d25a27c2692p-53}, {0x1.1835a88be7c13p-1, 0x1.c621cec00c301p-55},
    {0x1.0604e0fe4ef0fp0, -0x1.c8ae842ec057ap-54}, {0x1.4c124b2148e13p1, 0x1.a8d9ef8142b47p-53},
    {0x1.0f1d44c51b591p1, -0x1.465ab75a13c4fp-61}, {0x1.1e00babdefeb4p-1, -0x1.928df287a668fp-58},
    {0x1.031f57e54adbep0, 0x1.338b4259c0270p-54}, {0x1.4a9f8694c6d6bp1, 0x1.26f6d2c582f3bp-53},
    {0x1.109009519d639p1, 0x1.01398408cb59ep-54}, {0x1.23b71e2cc9e6ap-1, 0x1.c421c9f38224ep-57},
    {0x1.0044262dddde3p0, 0x1.c3bc53e5aaf7ap-55}, {0x1.4931edb91057ep1, -0x1.01dfb96df261ep-53},
    {0x1.11fda22d53e27p1, -0x1.568cb1c824fd8p-53}, {0x1.2958e59308e31p-1, -0x1.09e73b0c6c087p-56},
    {0x1.fae684f57cc00p-1, -0x1.46479c173e7afp-55}, {0x1.47c97bdf8098cp1, 0x1.dcfa54969a0bep-56},
    {0x1.13661406e3a18p1, 0x1.6bf44a37155f3p-53}, {0x1.2ee628406cbcap-1, 0x1.c5d5e9ff0cf8dp-55},
    {0x1.f559424818e66p-1, 0x1.bbbb718dfa201p-57}, {0x1.46662b3427a26p1, -0x1.5713174e7d7dcp-53},
    {0x1.14c964b23c97fp1, -0x1.015953e799e19p-53}, {0x1.345f01cce37bbp-1, 0x1.1021137c71102p-55},
    {0x1.efe068bba2275p-1, 0x1.24a3b2e61a70bp-55}, {0x1.4507f4d109f29p1, 0x1.d65a1e52297c6p-53},
    {0x1.16279b155a47bp1, -0x1.76344c4206ddfp-56}, {0x1.39c391cd4171ap-1, -0x1.2304331d8bf46p-55},
    {0x1.ea7bd8bb44317p-1, -0x1.506e0cffd1159p-56}, {0x1.43aed0d0f2752p1, -0x1.39b9200eae84fp-54},
    {0x1.1780bf1571c53p1, -0x1.bb8fdb2ec01cep-53}, {0x1.3f13fb89e96f4p-1, 0x1.ecf8b492644f0p-56},
    {0x1.e52b6efe9c33cp-1, 0x1.3e486c1959596p-55}, {0x1.425ab661c875bp1, 0x1.b986993df26d2p-54},
    {0x1.18d4d9849bc49p1, 0x1.95a09055ded43p-54}, {0x1.445065b795b56p-1, -0x1.f76d0163f79c8p-56},
    {0x1.dfef04d0efedbp-1, -0x1.9f0971d6f161cp-56}, {0x1.410b9bd65d643p1, -0x1.4d5ff94476980p-54},
    {0x1.1a23f41006d62p1, -0x1.b1bc6e93dc136p-53}, {0x1.4978fa3269ee1p-1, 0x1.2419a87f2a458p-56},
    {0x1.dac670561bb4fp-1, 0x1.a2b7f222f65e2p-55}, {0x1.3fc176b7a8560p1, -0x1.441a3bd3f1083p-58},
    {0x1.1b6e192ebbe44p1, 0x1.b1b466a88828ep-53}, {0x1.4e8de5bb6ec04p-1, 0x1.4a33dbeb3796cp-55},
    {0x1.d5b184cd16e2cp-1, 0x1.d521d4eea7d44p-56}, {0x1.3e7c3bd567217p1, 0x1.8faad86cefb58p-54},
    {0x1.1cb35410fd18dp1, 0x1.bf7c5126e18bdp-54}, {0x1.538f57b89061fp-1, -0x1.1bb74abda520cp-55},
    {0x1.d0b012cff5412p-1, -0x1.5f07ddbf9ebccp-56}, {0x1.3d3bdf561eb91p1, -0x1.9eafca1f50f76p-53},
    {0x1.1df3b09045814p1, -0x1.7379422d8ccffp-54}, {0x1.587d81f732fbbp-1, -0x1.5e5c9d8c5a950p-56},
    {0x1.cbc1e89152a76p-1, -0x1.1c0cead74734ap-55}, {0x1.3c0054c67612ap1, -0x1.b9d2091d2eecfp-53},
    {0x1.1f2f3b1fee27bp1, -0x1.3d34c431d0e4dp-54}, {0x1.5d58987169b18p-1, 0x1.0028e4bc5e7cap-57},
    {0x1.c6e6d2171bf18p-1, 0x1.f4ba8d3373e1bp-55}, {0x1.3ac98f27e8652p1, 0x1.0a5fd4e57fd8ap-53},
    {0x1.206600be7bd52p1, 0x1.3a677fc8d1900p-54}, {0x1.6220d115d7b8ep-1, -0x1.2b785350ee8c1p-57},
    {0x1.c21e9972adea3p-1, -0x1.805d24c938dc2p-55}, {0x1.399780fecce35p1, -0x1.a5cc2f3356adap-54},
    {0x1.21980ee797570p1, -0x1.8586539c6c089p-53}, {0x1.66d663923e087p-1, -0x1.6ea6febe8bbbap-56},
    {0x1.bd6906f6479aap-1, -0x1.13e7ba3e2ea15p-55}, {0x1.386a1c5fb34f7p1, -0x1.b7c8bcf6e8c82p-53},
    {0x1.22c57386b0eaep1, -0x1.41475c7e5d2e8p-54}, {0x1.6b798920b3d99p-1, -0x1.a80386188c50ep-55},
    {0x1.b8c5e167d1c98p-1, -0x1.19bd9c2741720p-58}, {0x1.374152fc15db2p1, 0x1.08c6896ed1a95p-54},
    {0x1.23ee3cea4e5f2p1, 0x1.233050127fcc0p-53}, {0x1.700a7c5784634p-1, -0x1.8c34d25aadef6p-56},
    {0x1.b434ee31013fdp-1, -0x1.0520d0701d877p-55}, {0x1.361d162e61b8bp1, 0x1.4be8fd7c9b7e6p-53},
    {0x1.251279b802819p1, 0x1.6eaa5d3534893p-55}, {0x1.748978fba8e0fp-1, 0x1.7b2a6165884a1p-59},
    {0x1.afb5f18cdcc22p-1, -0x1.e2eddfb3cd03cp-55}, {0x1.34fd570558995p1, -0x1.eb8a46545060cp-53},
    {0x1.263238e10ba10p1, -0x1.b38893871bfa8p-55}, {0x1.78f6bbd5d315ep-1, 0x1.406a089803740p-55},
    {0x1.ab48aeb2b28d2p-1, 0x1.e8b57b951019bp-56}, {0x1.33e2064ece0c1p1, -0x1.35b81ef4bb1c9p-53},
    {0x1.274d8997962e4p1, -0x1.22b44c415c42cp-53}, {0x1.7d528289fa093p-1, 0x1.560821e2f3aa9p-55},
    {0x1.a6ece7fe8b99dp-1, 0x1.bd7948ff2fac9p-56}, {0x1.32cb14a1c44f3p1, 0x1.c4e05ab888d5dp-53},
    {0x1.28647b449feb1p1, -0x1.d4cc5eea03524p-57}, {0x1.819d0b7158a4dp-1, -0x1.bf76229d3b917p-56},
    {0x1.a2a25f172cfe4p-1, -0x1.d700509dad6cep-56}, {0x1.31b87267eca85p1, 0x1.49449e13b4ca7p-55},
    {0x1.29771d7e7791fp1, 0x1.55426d44fb6e1p-53}, {0x1.85d69576cc2c5p-1, 0x1.6b66e7fc8b8c3p-57},
    {0x1.9e68d511b976bp-1, 0x1.d9eb0c63689ddp-55}, {0x1.30aa0fe68fc67p1, 0x1.d5fa58be83d55p-60},
    {0x1.2a857fffd473dp1, 0x1.a3e7a0186b990p-53}, {0x1.89ff5ff57f1f8p-1, -0x1.55b9a5e177a1bp-55},
    {0x1.9a400a9306839p-1, -0x1.d6064eeff375dp-57}, {0x1.2f9fdd46e309ap1, 0x1.6fd0cca9a3a8ep-53},
    {0x1.2b8fb29f8130ap1, 0x1.be16410227be5p-56}, {0x1.8e17aa99cc05ep-1, -0x1.ec182ab042f61p-56},
    {0x1.9627bfeeb99d3p-1, -0x1.aa5e488aa6084p-56}, {0x1.2e99ca9dcfd01p1, -0x1.50352ef163c1ap-54},
    {0x1.2c95c548946a4p1, -0x1.b051d3bd657e9p-53}, {0x1.921fb54442d18p-1, 0x1.1a62633145c07p-55},
    {0x1.921fb54442d18p-1, 0x1.1a62633145c07p-55}, {0x1.2d97c7f3321d2p1, 0x1.a79394c9e8a0ap-54},
    {0x1.2d97c7f3321d2p1, 0x1.a79394c9e8a0ap-54},
};

// Brings ax, ay into range with the same angle.
HM_ANGLE_FN void angle_rescale(double &ax, double &ay)
{
    const double s = ax + ay;
    if (s > 0x1p500) {
        const bool inf = !(ax < HUGE_VAL && ay < HUGE_VAL);
        ax = inf ? (ax < HUGE_VAL ? 0.0 : 1.0) : ax * 0x1p-600;
        ay = inf ? (ay < HUGE_VAL ? 0.0 : 1.0) : ay * 0x1p-600;
    } else if (s < 0x1p-500) {
        ax = s == 0.0 ? 1.0 : ax * 0x1p600;
        ay = ay * 0x1p600;
    }
}

// atan2(y, x); tab: kAtan.
HM_ANGLE_FN double angle_of(double y, double x, const AngleEntry *tab)
{
    double ax = fabs(x), ay = fabs(y);
    const double s = ax + ay;
    const bool odd = s < 0x1p-500 || s > 0x1p500;
#if defined(__HIP_DEVICE_COMPILE__)
    if (__builtin_expect(__any(odd), 0)) angle_rescale(ax, ay);
#else
    if (odd) angle_rescale(ax, ay);
#endif
    const bool swap = ay > ax;
    const double mx = swap ? ay : ax, mn = swap ? ax : ay;
#if defined(__HIP_DEVICE_COMPILE__)
    const double q = mn * __builtin_amdgcn_rcp(mx);
#else
    const double q = mn / mx;
#endif
    // q is 1 at most but for the reciprocal's 2^-20 or so: i is 64 at most, and 0 for NaN
    const uint32_t i = (uint32_t)fmax(fma(q, 64.0, 0.5), 0.0);
    const double c = (double)i * (1.0 / 64.0);
    const double num = fma(-c, mx, mn), den = fma(c, mn, mx);
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(den);
#else
    double r = (double)(1.0f / (float)den);
    if (!(r > 0.0 && r < HUGE_VAL)) r = 1.0 / den;
#endif
    r = fma(fma(-den, r, 1.0), r, r);
    double u = num * r;
    u = fma(fma(-u, den, num), r, u);
    const double z = u * u;
    const double p = fma(z, fma(z, -1.0 / 7, 1.0 / 5), -1.0 / 3);
    const double v = fma(u * z, p, u);
    // the octant's angle at c, and atan(u) to it or from it
    uint64_t xb, vb;
    memcpy(&xb, &x, sizeof xb);
    memcpy(&vb, &v, sizeof vb);
    const uint32_t neg = (uint32_t)(xb >> 32) & 0x80000000u, flip = neg ^ (swap ? 0x80000000u : 0u);
    const AngleEntry t = tab[4 * i + (neg >> 30) + (swap ? 1u : 0u)];
    vb ^= (uint64_t)flip << 32;
    double w;
    memcpy(&w, &vb, sizeof w);
    return copysign(t.hi + (t.lo + w), y);
}

#if defined(__HIPCC__)
// Fills a workgroup's table of angle_of in LDS; every thread takes part, before a
// barrier of the caller's.
__device__ __forceinline__ void fill_angle_table(AngleEntry *tab)
{
    for (int q = threadIdx.x; q < kAngleEntries; q += blockDim.x) tab[q] = kAtan[q];
}
#endif

}  // namespace hm
