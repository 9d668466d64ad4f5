// pw_core64.h -- the Gaussian core (rho^2 <= 90 sigma^2) of the FP64 kernels
// without exp, erf or branches.  Internal to libpawan_gpu.so.
//
// With s = rho^2/sigma^2, e = exp(-s/2), B(s) = sum_k s^k/(2k+5)!! and
// G = e B (the incomplete-gamma series of erf, A&S 6.5.29),
//   q = K (e/3 + s G) / sigma^3,   F = -3 K G / sigma^5,   Z = K e / sigma^3,
// K = (2 pi)^-3/2: sums of positive terms, so q and F keep their digits as
// rho -> 0, where the reference's phi/rho_bar - Z cancels.  G comes from 64
// pieces of degree 10 and e from the piece's exp(-s_c/2) times a degree-11
// polynomial (fit_core_table64.py beside this file; largest relative errors
// of the FP64 evaluation 2.4e-16 and 2.9e-16).  Rows are read per lane from
// LDS: 96 bytes in six 16-byte reads, 6 KB in all.
//
// The pairs within the core bound the FP64 sums of rings (sigma/R of 0.05-0.2
// puts a third to all of the pairs there): the library's exp and erf are
// about 150 instructions with a divergent branch in erf, this is 32 with
// none.  Measured on the LDS-tiled direct sum (k_pair_fp64, one item per 256
// targets): ring of 1,000 particles 404 -> 345 us per right-hand side, helix
// of 147,200 76.5 -> 68.2 ms, 48 independent rings 9.0 -> 7.5 ms; its error
// against 64-bit torch sums is no larger (rings 1.2e-13 -> 5.5e-14).
#pragma once

#include <hip/hip_runtime.h>

namespace pw {

constexpr int kCore64Pieces = 64;
constexpr int kCore64Row = 12;  // c0 .. c10, exp(-s_c/2)
constexpr double kCore64Width = 1.40625;          // 45/32: 64 pieces cover [0, 90]
constexpr double kCore64Scale = 32.0 / 45.0;
constexpr double kCore64K = 0x1.0411e71d77959p-4;  // (2 pi)^-3/2

static __constant__ double kCore64Exp[12] = {
    0x1.0000000000000p+0, 0x1.0000000000000p+0, 0x1.0000000000013p-1, 0x1.555555555555bp-3,
    0x1.555555554e4a0p-5, 0x1.111111110ee65p-7, 0x1.6c16c18a7bb0cp-10, 0x1.a01a01b2cd134p-13,
    0x1.a0198b14e6288p-16, 0x1.71ddf1666ae61p-19, 0x1.28ba085c55d89p-22, 0x1.af6a825a81c16p-26};
static __constant__ __align__(16) double kCore64Table[kCore64Pieces][kCore64Row] = {
    {0x1.aa1194294b6bap-5, -0x1.295b7a9e3af69p-6, 0x1.c7c9549508c38p-9, -0x1.ec2f14f82666fp-12, 0x1.9d5f58c71d6eap-15, -0x1.1cfb0c6fed762p-18, 0x1.4dc60ae327fa9p-22, -0x1.54118f990e068p-26, 0x1.32c3cfb5d3012p-30, -0x1.f1ff6fb179198p-35, 0x1.6d98e522e52cep-39, 0x1.683cab7c5a6efp-1},
    {0x1.0808f88eb2b68p-5, -0x1.5df16d6d9d782p-7, 0x1.0383938e018fap-9, -0x1.11f983a15b93cp-12, 0x1.c4b61989d8d6cp-16, -0x1.343d7a9311da0p-19, 0x1.65839de613051p-23, -0x1.696a6bb53efd6p-27, 0x1.43eeef4de8a7cp-31, -0x1.058594f490b41p-35, 0x1.7e3ebe02e71d9p-40, 0x1.64a91583f48ecp-2},
    {0x1.4fcd8a10fb8b0p-6, -0x1.a37a31b1abdaep-8, 0x1.2b87d67159cd3p-10, -0x1.34232ba004848p-13, 0x1.f3bbfff62c614p-17, -0x1.4f823453640d3p-20, 0x1.80ea630c4bb4cp-24, -0x1.81bdd2d4dacfbp-28, 0x1.574a40b5fa8ddp-32, -0x1.13839377b3898p-36, 0x1.90b432a59961ap-41, 0x1.611e969df99c8p-3},
    {0x1.b70478a7846dep-7, -0x1.0090d16d4a3c7p-8, 0x1.5ef23e5ed2d80p-11, -0x1.5e85053cf491fp-14, 0x1.164340cdc8a78p-17, -0x1.6fc0f5c52369bp-21, 0x1.a0c5fcfcc3495p-25, -0x1.9da24e69b14c4p-29, 0x1.6d3b0965b73f8p-33, -0x1.23385ec6d585ap-37, 0x1.a540e397082bap-42, 0x1.5d9d17afe0ca0p-4},
    {0x1.27549d9f904e2p-7, -0x1.40d4b9180678dp-9, 0x1.a20f7fe96d18cp-12, -0x1.93cba1e340a42p-15, 0x1.38ef56f4c69f3p-18, -0x1.963c6fd25ce09p-22, 0x1.c619f1a8167bfp-26, -0x1.bdd42ddb7dc3fp-30, 0x1.863df31a44413p-34, -0x1.34f008ef47997p-38, 0x1.bc3ab31183398p-43, 0x1.5a2481d9d9ca2p-5},
    {0x1.990bb5c21756dp-8, -0x1.9ab569b8803e8p-10, 0x1.fb1b62d15984ap-13, -0x1.d7b1d269e352dp-16, 0x1.63c3d8b70da22p-19, -0x1.c49cf4610922fp-23, 0x1.f233d44a42afep-27, -0x1.e340d05c8c89ap-31, 0x1.a2ed83049826bp-35, -0x1.49077c11c9362p-39, 0x1.d60930c26c728p-44, 0x1.56b4be7637919p-6},
    {0x1.237af9f56490ap-8, -0x1.0d6402463f8cep-10, 0x1.399e12a025a6ep-13, -0x1.17bd65f7c741cp-16, 0x1.995235de09fdfp-20, -0x1.fd15de329c90dp-24, 0x1.1362139cb573ep-27, -0x1.078ae5565ee44p-31, 0x1.c40a9ea78416bp-36, -0x1.5ff0f10246d10p-40, 0x1.f329f8bef89bep-45, 0x1.534db718dc936p-7},
    {0x1.aaeef4ce0ec96p-9, -0x1.6a53cbb90cd34p-11, 0x1.8c04b383503e7p-14, -0x1.5154ab86a3037p-17, 0x1.dd2589fdfd61cp-21, -0x1.214d3b447c408p-24, 0x1.33005b116faf2p-28, -0x1.216ab05dcae07p-32, 0x1.ea87d90145c66p-37, -0x1.7a39c1f0d6e19p-41, 0x1.0a1b28d23145ep-45, 0x1.4fef558ea8751p-8},
    {0x1.40c5ce581c922p-9, -0x1.f39e03b6e948dp-12, 0x1.fef8c3596f1b6p-15, -0x1.9e0a80db32dc7p-18, 0x1.1a176b35100b1p-21, -0x1.4c94b13e19eb5p-25, 0x1.596a318cb9090p-29, -0x1.403933a0b12cfp-33, 0x1.0bcc45989fd57p-37, -0x1.98920fab559fbp-42, 0x1.1cf53805dfb41p-46, 0x1.4c9983dce7363p-9},
    {0x1.ed77311e414b1p-10, -0x1.60f1e9ab6b2c0p-12, 0x1.510116c885b0ep-15, -0x1.02e44fa623c16p-18, 0x1.52b284c2c0deep-22, -0x1.831c8a2bddd2ep-26, 0x1.88911826b3ba1p-30, -0x1.653b41aaa58c1p-34, 0x1.2662916c6392bp-38, -0x1.bbd6dc50780c6p-43, 0x1.329774b84cd14p-47, 0x1.494c2c40c1c86p-10},
    {0x1.83b0daac3210cp-10, -0x1.fe67f408fe308p-13, 0x1.c680122ac7489p-16, -0x1.4a1e30e02fe83p-19, 0x1.9d59cedfa3ddfp-23, -0x1.c8aa7db9b0097p-27, 0x1.c3120092807bdp-31, -0x1.921b8372a4168p-35, 0x1.460351d2d26b2p-39, -0x1.e51f7c76640d8p-44, 0x1.4b92892c48503p-48, 0x1.4607392eb013cp-11},
    {0x1.3666bd30ada4bp-10, -0x1.7939809437341p-13, 0x1.3941c0233ae76p-16, -0x1.ad68230454462p-20, 0x1.0098565559171p-23, -0x1.1140ccc3cff49p-27, 0x1.063c64ea709e9p-31, -0x1.c90f454846fc3p-36, 0x1.6bf6167330d78p-40, -0x1.0ae7cbc241280p-44, 0x1.689ba4462ec4cp-49, 0x1.42ca9551ec643p-12},
    {0x1.f96f514477455p-11, -0x1.1c819032f90f5p-13, 0x1.b910e5415839ep-17, -0x1.1cf0b2fae06f5p-20, 0x1.444c007021698p-24, -0x1.4c05b2ec7d81fp-28, 0x1.34d0905910a10p-32, -0x1.06850ab88b57cp-36, 0x1.99e742c69ee89p-41, -0x1.27d7b645b1c2ap-45, 0x1.8a9745486a7c7p-50, 0x1.3f962b8be83bfp-13},
    {0x1.a1a2ceeb7f822p-11, -0x1.b5336718eed09p-14, 0x1.3cdb7f1b617a6p-17, -0x1.81c15428e5930p-21, 0x1.a166b54c30950p-25, -0x1.99e97b9096254p-29, 0x1.70a15048ae6f0p-33, -0x1.31035a91b0961p-37, 0x1.d20bb682c4307p-42, -0x1.4a866155bb163p-46, 0x1.b2a7a26e0a61ap-51, 0x1.3c69e6f3c287ep-14},
    {0x1.5d9e711da1eecp-11, -0x1.55a41480e4259p-14, 0x1.d0036ac5b0d4ep-18, -0x1.0a3f0c3a69243p-21, 0x1.119a974d9d5f7p-25, -0x1.013f1d55d138ep-29, 0x1.be5e85e8ac24cp-34, -0x1.66b77608de70ap-38, 0x1.0ba93e0ae79f7p-42, -0x1.7473f5a2d517ep-47, 0x1.e23ffe20c5296p-52, 0x1.3945b2d5bf322p-15},
    {0x1.2812244dfb36bp-11, -0x1.0f1218a2b8fe3p-14, 0x1.59d7adaa2abfcp-18, -0x1.76796d60a20afp-22, 0x1.6d50c27533694p-26, -0x1.485ebffe3ca85p-30, 0x1.1251087731799p-34, -0x1.ab5832a103447p-39, 0x1.36d53ee12a3a2p-43, -0x1.a798d63bd5e9fp-48, 0x1.0d9f630786ed0p-52, 0x1.36297ab2c00f2p-16},
    {0x1.fa97ecabb3deap-12, -0x1.b41bb591dfb5bp-15, 0x1.0607cb1fdfe0dp-18, -0x1.0c16a54bb447bp-22, 0x1.f09c723bb5b46p-27, -0x1.aa5aea08d1e36p-31, 0x1.5666c3672e888p-35, -0x1.0204e9a156f2dp-39, 0x1.6d32816453b58p-44, -0x1.e690806af616ep-49, 0x1.30088c62c0961p-53, 0x1.33152a3fbf226p-17},
    {0x1.b55b79e20020bp-12, -0x1.632ea632d8008p-15, 0x1.9316c2afb9f7ap-19, -0x1.865cbba652cfbp-23, 0x1.577b0912254bcp-27, -0x1.1986d222dd517p-31, 0x1.b22a3865e0f4dp-36, -0x1.3bfd2bf94a851p-40, 0x1.b260e6cd7d93ap-45, -0x1.1a6aa947d84b5p-49, 0x1.59f1b1e5e4607p-54, 0x1.3008ad654a370p-18},
    {0x1.7ca89d69563c5p-12, -0x1.248498cb8c260p-15, 0x1.3a591882000ecp-19, -0x1.20b5200566f93p-23, 0x1.e325630825775p-28, -0x1.7a0e8653a1d90p-32, 0x1.17aae83a09767p-36, -0x1.88a332c4c3020p-41, 0x1.05adf45a8db8dp-45, -0x1.4b8a39221ff0fp-50, 0x1.8d722e1a89341p-55, 0x1.2d03f03effc8ap-19},
    {0x1.4dbb1f7fff092p-12, -0x1.e6b254dc0d45cp-16, 0x1.f0812dce837ddp-20, -0x1.b1570ce9fd1f9p-24, 0x1.593e9a63a09bfp-28, -0x1.020297928130fp-32, 0x1.6e0d4e052f771p-37, -0x1.ef2563bcc784fp-42, 0x1.3f85a934a9bb4p-46, -0x1.89d22ac70655fp-51, 0x1.cd50eba34e715p-56, 0x1.2a06df1b0d397p-20},
    {0x1.2683efdd81502p-12, -0x1.9898c4f68cc67p-16, 0x1.8ca56383d87b2p-20, -0x1.49a5b3159b167p-24, 0x1.f4dca45110ab7p-29, -0x1.65bdcd14503ddp-33, 0x1.e6ac73155ec7ep-38, -0x1.3ce65a3a0f967p-42, 0x1.8b8aad9eab2f7p-47, -0x1.d996aa96ce027p-52, 0x1.0ea2955c35286p-56, 0x1.27116679ae527p-21},
    {0x1.0575326e4c7f1p-12, -0x1.59e20149aa8f0p-16, 0x1.4038874e0d55ap-20, -0x1.fbd842c67aa46p-25, 0x1.70757b9f00c4dp-29, -0x1.f78890f912425p-34, 0x1.48818a05228b5p-38, -0x1.9bb974ec1b3e1p-43, 0x1.f088d5ad66296p-48, -0x1.2066bd4e4b5c1p-52, 0x1.4128b9acd7157p-57, 0x1.2423730cae0a1p-22},
    {0x1.d2bd34ee5306cp-13, -0x1.27036791870b6p-16, 0x1.05055cd57f02cp-20, -0x1.8bb97a1093abbp-25, 0x1.12a4902cb12e5p-29, -0x1.67773c4552f6ep-34, 0x1.c21a20240616bp-39, -0x1.0f6d55f154fabp-43, 0x1.3c133918019fdp-48, -0x1.63dddddb6b8cbp-53, 0x1.81a20afdff707p-58, 0x1.213cf1b6e88e3p-23},
    {0x1.a2a9274e6b1f1p-13, -0x1.fabc8a7598e6dp-17, 0x1.ad4da073cb839p-21, -0x1.37a84587b1824p-25, 0x1.9e78e4f98f718p-30, -0x1.041a2fb4d3722p-34, 0x1.38c6367a271bcp-39, -0x1.6b1217efca0ccp-44, 0x1.981939d0ae888p-49, -0x1.bcf8ec9620e13p-54, 0x1.d4b6ef6dc1186p-59, 0x1.1e5dcf8bce8e3p-24},
    {0x1.793d60cc54c1ep-13, -0x1.b5f819f9ae38cp-17, 0x1.63ea57a2bf889p-21, -0x1.efbefe870a830p-26, 0x1.3c545686ccb3dp-30, -0x1.7d37727d21bcap-35, 0x1.b8a415fdf7c77p-40, -0x1.ec81ed740ff6dp-45, 0x1.0b258032daeeap-49, -0x1.19eebf1695da7p-54, 0x1.2069dc5d4234bp-59, 0x1.1b85f9cee9c21p-25},
    {0x1.55561f066677bp-13, -0x1.7cbf57ea11487p-17, 0x1.2949bbd6f2bacp-21, -0x1.8de255690c16fp-26, 0x1.e7fe100f467abp-31, -0x1.1ab57e808b0fap-35, 0x1.3a6cd68806038p-40, -0x1.5296ef867b7acp-45, 0x1.628f7cf455c52p-50, -0x1.6a0e12555c9aep-55, 0x1.67725bc001339p-60, 0x1.18b55df362ab7p-26},
    {0x1.360a65f0d76d5p-13, -0x1.4cc9e946602c3p-17, 0x1.f41490c869a21p-22, -0x1.4209d5edd639dp-26, 0x1.7c219ce347f59p-31, -0x1.a80354f7776e8p-36, 0x1.c63dbe7a53df3p-41, -0x1.d79ebb4a0532ap-46, 0x1.dcdf96fc9cfbdp-51, -0x1.d71f3c244dc7cp-56, 0x1.c5b34447a43a9p-61, 0x1.15ebe99b878d6p-27},
    {0x1.1a9e8386dc0e4p-13, -0x1.24532172f8b36p-17, 0x1.a74e216eb0f47p-22, -0x1.06b183da84e71p-26, 0x1.2ad65ab74059fp-31, -0x1.414e6b0720342p-36, 0x1.4beb601ca69edp-41, -0x1.4c8baf873fff6p-46, 0x1.44d72f87c3cdap-51, -0x1.368589c228f19p-56, 0x1.21fca9d3f3125p-61, 0x1.13298a9854973p-28},
    {0x1.027a04f35674cp-13, -0x1.01f8f64eb4827p-17, 0x1.68748d42207f7p-22, -0x1.afb0fd4d55e6ep-27, 0x1.d9e33c8fb9ca0p-32, -0x1.ebbb3c14ca99ep-37, 0x1.ea5eba591df9ap-42, -0x1.da828c35009f9p-47, 0x1.c01076ebacdf1p-52, -0x1.9e8bec423ec54p-57, 0x1.776114e382526p-62, 0x1.106e2ee8fd40cp-29},
    {0x1.da404e2e8eb2bp-14, -0x1.c9480f9ed84a3p-18, 0x1.34a47572f4367p-22, -0x1.651ce15da7733p-27, 0x1.7abee40089f4dp-32, -0x1.7bbaa3c2e4b67p-37, 0x1.6df2f99daf50dp-42, -0x1.565535f59c2aap-47, 0x1.38b2e51254270p-52, -0x1.18200503cc546p-57, 0x1.ebf413480702fp-63, 0x1.0db9c4ba76d37p-30},
    {0x1.b4542cddf72f8p-14, -0x1.96ec147c2f0a2p-18, 0x1.09a5d53972601p-22, -0x1.294a61e4ee1b0p-27, 0x1.30f81f69445b0p-32, -0x1.27c1fe573ae54p-37, 0x1.13bb9d8417219p-42, -0x1.f32ef63abefa2p-48, 0x1.b96ba3e43d1c1p-53, -0x1.7f16e68558d6fp-58, 0x1.46470e63a4d1ep-63, 0x1.0b0c3a67041e7p-31},
    {0x1.9285094af1f8fp-14, -0x1.6b7978728c71dp-18, 0x1.cb80c95841482p-23, -0x1.f1e9f9ad77161p-28, 0x1.ee910d9f00fe3p-33, -0x1.d06c5f79e408ap-38, 0x1.a348f7521adb9p-43, -0x1.6f980826ea8cfp-48, 0x1.3aef811c22bbcp-53, -0x1.08f1e848da51cp-58, 0x1.b5e578ddc911ap-64, 0x1.08657e75c251fp-32},
    {0x1.744479764ee89p-14, -0x1.45d045633761dp-18, 0x1.8f380607ff086p-23, -0x1.a347e96323854p-28, 0x1.93a6c54c6058cp-33, -0x1.6f65881897abcp-38, 0x1.41821364fdac4p-43, -0x1.1140674e64d63p-48, 0x1.c600f809ff87cp-54, -0x1.727b85f39a448p-59, 0x1.2933178170b23p-64, 0x1.05c57f9a36ff7p-33},
    {0x1.591aed6a0450ap-14, -0x1.25064d8d01369p-18, 0x1.5c5333d251dbfp-23, -0x1.62e8df92efd98p-28, 0x1.4b7b683595398p-33, -0x1.24b54350270c4p-38, 0x1.f1076b9b18580p-44, -0x1.99decbb3e223dp-49, 0x1.4a6dc73cde048p-54, -0x1.05bc556d412ecp-59, 0x1.97d881f039c65p-65, 0x1.032c2cb3df3b8p-34},
    {0x1.40a379735090cp-14, -0x1.085be80553d71p-18, 0x1.312412980fccap-23, -0x1.2de5c7b10640dp-28, 0x1.11cc0f30f4345p-33, -0x1.d587cb1caa570p-39, 0x1.8318e886a079ap-44, -0x1.35fd3bc586bfcp-49, 0x1.e56bb4b31e361p-55, -0x1.757fb6ce7cd07p-60, 0x1.1aca5aa6d7160p-65, 0x1.009974cdbfdecp-35},
    {0x1.2a887f1e9ce5ap-14, -0x1.de668d96d2200p-19, 0x1.0c52d52116e96p-23, -0x1.01fe5c8404012p-28, 0x1.c6c7399d2e474p-34, -0x1.7af6ce3ae4e36p-39, 0x1.2fa2e3e3ec4cfp-44, -0x1.d8a207ba09824p-50, 0x1.67ad4fc218e5bp-55, -0x1.0d0459d09f852p-60, 0x1.8c1d7b8e21626p-66, 0x1.fc1a8e3bedc4cp-37},
    {0x1.16810230d04ddp-14, -0x1.b2137ebaaef84p-19, 0x1.d995eced30225p-24, -0x1.bae0cd5efaba4p-29, 0x1.7ba5d75069c1ep-34, -0x1.33b131a32c091p-39, 0x1.df8f5186d48fdp-45, -0x1.6b05b98909d28p-50, 0x1.0cb774c73e0aep-55, -0x1.870405cd0d3a8p-61, 0x1.1819acf44d24ap-66, 0x1.f70f260a9bac8p-38},
    {0x1.044e83707a5b1p-14, -0x1.8ae517b3f5b09p-19, 0x1.a3595f74f8707p-24, -0x1.7db368c32072dp-29, 0x1.3e7ac6cf34589p-34, -0x1.f6783240fadbap-40, 0x1.7d20c89984949p-45, -0x1.18d2a71ae3fb7p-50, 0x1.94ad829fb1f65p-56, -0x1.1e9a84d14ae09p-61, 0x1.8fc589fbd799dp-67, 0x1.f210901d9ada9p-39},
    {0x1.e77688974eefep-15, -0x1.682555b8fa71fp-19, 0x1.7483b4dc5e1bdp-24, -0x1.4a438e24bafbcp-29, 0x1.0c67a1dfdc77dp-34, -0x1.9c77a1517cf28p-40, 0x1.30bc52f7b8247p-45, -0x1.b5699b412caf6p-51, 0x1.32fd7308e3768p-56, -0x1.a790bd4fa7b95p-62, 0x1.1fc9da75c43c1p-67, 0x1.ed1eabdea43afp-40},
    {0x1.c931ba74c22c4p-15, -0x1.493b36ac8dec2p-19, 0x1.4beac157b1ec9p-24, -0x1.1ed233997e684p-29, 0x1.c6653fa2d78f0p-35, -0x1.544ddc54103dep-40, 0x1.ea1ccd9654cc8p-46, -0x1.56d8fa6148dd8p-51, 0x1.d511f6d947358p-57, -0x1.3b69ae840ad1bp-62, 0x1.a1d018d5fe705p-68, 0x1.e839590a43a19p-41},
    {0x1.ad7e2ba9e6df2p-15, -0x1.2da584d83ac33p-19, 0x1.289932659ff25p-24, -0x1.f3f20025c2c27p-30, 0x1.823d828eb6725p-35, -0x1.1a1e94f225d33p-40, 0x1.8c4834222e250p-46, -0x1.0e5e027f22624p-51, 0x1.68c700b2a9e43p-57, -0x1.d9369c8955b04p-63, 0x1.31b5b24fa83d5p-68, 0x1.e36077af0548ap-42},
    {0x1.9415e2d16f152p-15, -0x1.14f6ab38d9000p-19, 0x1.09c4304939996p-24, -0x1.b52e298cf95e8p-30, 0x1.499c980e46806p-35, -0x1.d5e9160affdbap-41, 0x1.42147ff1610fdp-46, -0x1.ace5569ccfbadp-52, 0x1.174418a615907p-57, -0x1.6578d209b44a5p-63, 0x1.c2c587ed7f559p-69, 0x1.de93e82ca565cp-43},
    {0x1.7cbbcb7863b21p-15, -0x1.fda2b1fbda812p-20, 0x1.dd8670c8c8e90p-25, -0x1.7f84ab7a593bdp-30, 0x1.1a59810b3434ep-35, -0x1.890f63f812653p-41, 0x1.071144f0a71fbp-46, -0x1.5611f3e5614b8p-52, 0x1.b2fbdad55e47dp-58, -0x1.0fd880d2a7556p-63, 0x1.4ebe8640e0c2ap-69, 0x1.d9d38b3341d13p-44},
    {0x1.673a67d2fb25cp-15, -0x1.d5cb909af694fp-20, 0x1.ae13596606f2ep-25, -0x1.517821f27c5fap-30, 0x1.e57917b94b7e1p-36, -0x1.4a257b38d5cfdp-41, 0x1.afc31b452773dp-47, -0x1.12429c401959ep-52, 0x1.54bd370e4fcbbp-58, -0x1.a0191823c4d97p-64, 0x1.f49b7361f830fp-70, 0x1.d51f41c28db92p-45},
    {0x1.5362b9d1c5cb7p-15, -0x1.b1df0cdf1ed48p-20, 0x1.84436aaf9657cp-25, -0x1.29d0611f2b2b5p-30, 0x1.a2cc6fdfee166p-36, -0x1.166780e7a53a9p-41, 0x1.63e99ae0e64c5p-47, -0x1.b9ffaf6e07edfp-53, 0x1.0c6615ef2a1cdp-58, -0x1.40637bfcd3393p-64, 0x1.78cdbe9461d84p-70, 0x1.d076ed29075c5p-46},
    {0x1.410b596b69b46p-15, -0x1.9167463a81776p-20, 0x1.5f50527726293p-25, -0x1.078cb69e637c6p-30, 0x1.6a782268d7135p-36, -0x1.d7533a41c5c3fp-42, 0x1.26a66b67ccbd0p-47, -0x1.65e06174a62fap-53, 0x1.a914c6d8c9ddep-59, -0x1.f042d6fd38906p-65, 0x1.1d6964ee06600p-70, 0x1.cbda6f032fc74p-47},
    {0x1.300faffa511d0p-15, -0x1.73fe64e78a79ap-20, 0x1.3e92892eec644p-25, -0x1.d3b23e45ac3b4p-31, 0x1.3ab4016ea3c5bp-36, -0x1.9069e75727c86p-42, 0x1.e9df72de9e0b3p-48, -0x1.2318f8b07b50cp-53, 0x1.5253979529e8ap-59, -0x1.827aa3f650281p-65, 0x1.b2fd675ea4319p-71, 0x1.c749a93ac48d5p-48},
    {0x1.204f522713e67p-15, -0x1.594c22ea335d4p-20, 0x1.217c032944267p-25, -0x1.a00b83e71b5a4p-31, 0x1.120deec33572dp-36, -0x1.555a6c1483ebcp-42, 0x1.98d349a64ab73p-48, -0x1.dba4f7f0706adp-54, 0x1.0e96ae44c96b8p-59, -0x1.2e9691c852fd5p-65, 0x1.4d669545cd703p-71, 0x1.c2c47e05fb7b5p-49},
    {0x1.11ad731a90804p-15, -0x1.4103c0c80ca59p-20, 0x1.0793e260e8996p-25, -0x1.73005d6d162cfp-31, 0x1.deb0887382d40p-37, -0x1.23f9255f1f768p-42, 0x1.567991fce7692p-48, -0x1.863beea2bd3d9p-54, 0x1.b2d8481ef1eaep-60, -0x1.dc3c5c4c8c43dp-66, 0x1.00f4e79b1d90ep-71, 0x1.be4acfe6c03b6p-50},
    {0x1.04106cb18e13ep-15, -0x1.2ae251d215888p-20, 0x1.e0e5e89c4dcb1p-26, -0x1.4b9bf3510b83ep-31, 0x1.a33831ae9005dp-37, -0x1.f5118726743d2p-43, 0x1.1fee7cfb0aa18p-48, -0x1.4174e5cfc979ep-54, 0x1.5ef7ee853a947p-60, -0x1.789adbe8f404bp-66, 0x1.8e30dcf185c39p-72, 0x1.b9dc81a9f3e82p-51},
    {0x1.eec2b26cecd3ep-16, -0x1.16ad4ff0bef25p-20, 0x1.b781a5ac0f7b4p-26, -0x1.2910d40314035p-31, 0x1.701cf6b5e1baap-37, -0x1.af457f3149a16p-43, 0x1.e5d530029f25bp-49, -0x1.09d46f892aacdp-54, 0x1.1c7cd20651d59p-60, -0x1.2b38054adac6dp-66, 0x1.361add40639cap-72, 0x1.b5797666ae883p-52},
    {0x1.d717778f6945cp-16, -0x1.04316a141bd20p-20, 0x1.9263106a2ea60p-26, -0x1.0ab1fff15f980p-31, 0x1.440fe810b03e6p-37, -0x1.744a5858b7197p-43, 0x1.9b3f119a88e90p-49, -0x1.b94c97e9cece3p-55, 0x1.cf1a2ec78fb6fp-61, -0x1.dd9e4434ed381p-67, 0x1.e5623dff18477p-73, 0x1.b121917d826e3p-53},
    {0x1.c0fa6a26af995p-16, -0x1.e68305da460e9p-21, 0x1.7107392803c19p-26, -0x1.dfda94c38e35dp-32, 0x1.1dfb9417cbb55p-37, -0x1.4249301a57141p-43, 0x1.5d3a725852b2ap-49, -0x1.6f9c66fa22f1cp-55, 0x1.7a6ce055162f2p-61, -0x1.7ed921a8acd86p-67, 0x1.7da986a5828acp-73, 0x1.acd4b697c1780p-54},
    {0x1.ac4a84f3021dep-16, -0x1.c76baf21c4df9p-21, 0x1.52fcf26f271f7p-26, -0x1.b08d91dc11bbdp-32, 0x1.f9f2a15af4684p-38, -0x1.17c2143e4a310p-43, 0x1.297aa26078becp-49, -0x1.3348e0126cdc7p-55, 0x1.36696875e521bp-61, -0x1.342a86723a75fp-67, 0x1.2d782a00fd06cp-73, 0x1.a892c9a6c4291p-55},
    {0x1.98ea0bf841061p-16, -0x1.aad68e739bb3dp-21, 0x1.37e222ac0c055p-26, -0x1.86aa35c39532ep-32, 0x1.c091557a8b8c5p-38, -0x1.e6f579ab76d91p-44, 0x1.fc4dbd54cf58dp-50, -0x1.01b655af5514ap-55, 0x1.ff1dbb5dfbeb0p-62, -0x1.f21a398f92e04p-68, 0x1.de5669914bfafp-74, 0x1.a45baee33299ep-56},
    {0x1.86be2b4f486acp-16, -0x1.90856d39f288bp-21, 0x1.1f61879e9548fp-26, -0x1.617cbb1c87380p-32, 0x1.8e910b8dd981cp-38, -0x1.a8e1e1b159d5dp-44, 0x1.b383d9bd49d47p-50, -0x1.b1a8bc157b7b1p-56, 0x1.a6492ef883d58p-62, -0x1.941d51f872d01p-68, 0x1.7d163a61a82cap-74, 0x1.a02f4acc4f39ap-57},
    {0x1.75aea2b1624b3p-16, -0x1.7841149567b9ep-21, 0x1.0930d7142bb14p-26, -0x1.406b578afefc1p-32, 0x1.62e320f8ecfd6p-38, -0x1.739f83adfe82dp-44, 0x1.762e54bfdceb2p-50, -0x1.6dfdf28945832p-56, 0x1.5e15e631fa46ep-62, -0x1.49168e5a9a688p-68, 0x1.30d7d33091670p-74, 0x1.9c0d8227435bep-58},
    {0x1.65a57be28d0c6p-16, -0x1.61d868c27643cp-21, 0x1.ea1e58cf384dap-27, -0x1.22f21b7d87719p-32, 0x1.3ca38fa56b6b2p-38, -0x1.45cdfb1a8ff32p-44, 0x1.42578a5cdaf37p-50, -0x1.35cde01a75e08p-56, 0x1.232f9eafa5bdep-62, -0x1.0cf551da9f59ap-68, 0x1.e99ee53482117p-75, 0x1.97f639fe6d8eap-59},
    {0x1.568eca6b82414p-16, -0x1.4d1fa4ff47796p-21, 0x1.c5876ad223a62p-27, -0x1.089f88486e1c3p-32, 0x1.1b11a2d966178p-38, -0x1.1e48b3de6b7fbp-44, 0x1.16664e2735e09p-50, -0x1.06ff478529882p-56, 0x1.e5eed1392e834p-63, -0x1.b9299f25fbc40p-69, 0x1.8ab0842207d2bp-75, 0x1.93e957a0b1b3dp-60},
    {0x1.485873535013cp-16, -0x1.39efb2dda3ce4p-21, 0x1.a43927a47eda7p-27, -0x1.e2237555e6589p-33, 0x1.fb1408dcbda23p-39, -0x1.f837f2b4de383p-45, 0x1.e217600bbc675p-51, -0x1.bfc3f9443b153p-57, 0x1.96b5bbd38ddb4p-63, -0x1.6b079e59fc286p-69, 0x1.3f542e825df55p-75, 0x1.8fe6c0a0cad9ep-61},
    {0x1.3af1fbbc76e9fp-16, -0x1.282598c9a9e10p-21, 0x1.85dbd4d7a40abp-27, -0x1.b7e81d28eb9e7p-33, 0x1.c703bceed7c8bp-39, -0x1.bcf8532213b08p-45, 0x1.a26926711a7a3p-51, -0x1.7e3217a22d09fp-57, 0x1.556a023817a16p-63, -0x1.2bb4ff2ff538ep-69, 0x1.034575db7b363p-75, 0x1.8bee5ad49eceep-62},
    {0x1.2e4c5d74d265ep-16, -0x1.17a1fc426fd53p-21, 0x1.6a221d4a0f08dp-27, -0x1.91fa4ca2af04ep-33, 0x1.9905b74ad50ffp-39, -0x1.897d34c1f6a87p-45, 0x1.6bfc7d9410f47p-51, -0x1.47135e6fb12edp-57, 0x1.1f6cbca331d91p-63, -0x1.f06ab1c226addp-70, 0x1.a675743607743p-76, 0x1.88000c54936a5p-63},
    {0x1.2259e0abb9802p-16, -0x1.0848b4d5a6cc6p-21, 0x1.50c7b153faa3dp-27, -0x1.6fda86faecd72p-33, 0x1.704fb79e1302ap-39, -0x1.5ca7afc1bb284p-45, 0x1.3d5a82652ddafp-51, -0x1.189bea34b3e07p-57, 0x1.e54aa0abc48d3p-64, -0x1.9c5ea85b4c546p-70, 0x1.59518bbdc2fffp-76, 0x1.841bbb7ae5881p-64},
    {0x1.170dfa1ffe91fp-16, -0x1.f400dad213630p-22, 0x1.39901a2313a2cp-27, -0x1.5119c6e66a475p-33, 0x1.4c34755a3890fp-39, -0x1.3585ec62c99a2p-45, 0x1.154c4e49b02aap-51, -0x1.e2a8fec98c3cep-58, 0x1.9ac9f958aa822p-64, -0x1.57900f0037df7p-70, 0x1.1b2b3a687da9fp-76, 0x1.80414ee301b1bp-65},
};

// the table into LDS (tab holds kCore64Pieces * kCore64Row doubles, 16-byte
// aligned) by a block of kThreads; the caller synchronises the block
// afterwards.  All loads are issued before the first is waited for: one after
// another they were 3 of the latencies that a small right-hand side consists of
// (1,000 particles: 12.25 us against 12.45).
template <int kThreads>
__device__ __forceinline__ void stage_core64(double* tab) {
  constexpr int kPairs = kCore64Pieces * kCore64Row / 2;
  static_assert(kCore64Row % 2 == 0, "16-byte pieces of a row");
  const double2* src = reinterpret_cast<const double2*>(&kCore64Table[0][0]);
  const int t = static_cast<int>(threadIdx.x);
  constexpr int kLoads = (kPairs + kThreads - 1) / kThreads;
  double2 v[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) v[i] = src[min(t + i * kThreads, kPairs - 1)];
#pragma unroll
  for (int i = 0; i < kLoads; ++i)
    if (t + i * kThreads < kPairs) reinterpret_cast<double2*>(tab)[t + i * kThreads] = v[i];
}

// e = exp(-s/2) and G(s), 0 <= s <= 90 (any other s, NaN included, reads a
// row of the table and returns a meaningless value)
__device__ __forceinline__ void core64(double s, const double* __restrict__ tab, double& e, double& g) {
  const int k = min(max(static_cast<int>(s * kCore64Scale), 0), kCore64Pieces - 1);
  const double2* __restrict__ row = reinterpret_cast<const double2*>(tab + kCore64Row * k);
  const double2 r0 = row[0], r1 = row[1], r2 = row[2], r3 = row[3], r4 = row[4], r5 = row[5];
  const double t = fma(-kCore64Width, static_cast<double>(k) + 0.5, s);
  g = fma(r5.x, t, r4.y);
  g = fma(g, t, r4.x);
  g = fma(g, t, r3.y);
  g = fma(g, t, r3.x);
  g = fma(g, t, r2.y);
  g = fma(g, t, r2.x);
  g = fma(g, t, r1.y);
  g = fma(g, t, r1.x);
  g = fma(g, t, r0.y);
  g = fma(g, t, r0.x);
  const double x = -0.5 * t;
  double p = kCore64Exp[11];
#pragma unroll
  for (int j = 10; j >= 0; --j) p = fma(p, x, kCore64Exp[j]);
  e = r5.y * p;
}

}  // namespace pw
