// x^y for normal x > 0 and |y log2 x| < 2^24, as 2^(y log2 x) with the
// logarithm held in two doubles (table-driven, after P. T. P. Tang's method of
// splitting the argument by a table of reciprocals): log2 x = e - log2(c_i) +
// log2(1 + r), r = c_i m - 1, |r| < 1/128, and 2^z = 2^k 2^(j/64) 2^f.
// About 50 instructions where the library's pow takes 250, which is what the
// contact-point solve's chain consisted of. Error against exact powers over
// x in [1e-12, 1e3], y in [-2, 6] (the solve's: a blockiness of 2 to 8 less two,
// n1 / n2, and that less two): at most 0.52 units in the last place (the
// library's pow: 1.33; the product of an integer and a fractional power that
// it replaces: 4.69).
#pragma once

#include <hip/hip_runtime.h>

namespace sqd {

// {1/m_i, -log2(1/m_i) rounded to 2^-42, the rest, 0} for the 128 slices of [1, 2)
static __device__ const double kPowLog[128 * 4] = {
    0x1.0000000000000p+0, 0x0.0p+0, 0x0.0p+0, 0.0,
    0x1.fa11caa01fa12p-1, 0x1.1363117a90000p-6, 0x1.ec0a3ae7eef8dp-44, 0.0,
    0x1.f6310aca0dbb5p-1, 0x1.c9363ba850000p-6, 0x1.f37b86dc20b16p-47, 0.0,
    0x1.f25f644230ab5p-1, 0x1.3ed3094688000p-5, -0x1.2ec59e20a3645p-44, 0.0,
    0x1.ee9c7f8458e02p-1, 0x1.985bfc3498000p-5, -0x1.7369f6f10b400p-44, 0.0,
    0x1.eae807aba01ebp-1, 0x1.f138983328000p-5, -0x1.6314fa37912c4p-44, 0.0,
    0x1.e741aa59750e4p-1, 0x1.24b5b7e134000p-4, 0x1.a41681fde8c44p-44, 0.0,
    0x1.e3a9179dc1a73p-1, 0x1.507b836034000p-4, -0x1.1189711531d93p-46, 0.0,
    0x1.e01e01e01e01ep-1, 0x1.7beee96b8c000p-4, -0x1.d7eaca90a689fp-44, 0.0,
    0x1.dca01dca01dcap-1, 0x1.a7111df348000p-4, 0x1.25009667e0d9dp-46, 0.0,
    0x1.d92f2231e7f8ap-1, 0x1.d1e34e35b8000p-4, 0x1.6b4d5164df95fp-47, 0.0,
    0x1.d5cac807572b2p-1, 0x1.fc66a0f0b0000p-4, 0x1.494ec4f791811p-49, 0.0,
    0x1.d272ca3fc5b1ap-1, 0x1.134e1b4890000p-3, 0x1.8c2a0a578e24dp-45, 0.0,
    0x1.cf26e5c44bfc6p-1, 0x1.284294b07a000p-3, 0x1.900ea58888daap-45, 0.0,
    0x1.cbe6d9601cbe7p-1, 0x1.3d1146d9a8000p-3, 0x1.4c5efccef202fp-44, 0.0,
    0x1.c8b265afb8a42p-1, 0x1.51bab907a6000p-3, -0x1.bad5e2a9da872p-46, 0.0,
    0x1.c5894d10d4986p-1, 0x1.663f6fac92000p-3, -0x1.9d62e501bd030p-44, 0.0,
    0x1.c26b5392ea01cp-1, 0x1.7a9fec7d06000p-3, -0x1.10084bd08319bp-46, 0.0,
    0x1.bf583ee868d8bp-1, 0x1.8edcae8352000p-3, 0x1.6d66225cf27b5p-44, 0.0,
    0x1.bc4fd65883e7bp-1, 0x1.a2f632320c000p-3, -0x1.e4ecc8c3be907p-45, 0.0,
    0x1.b951e2b18ff23p-1, 0x1.b6ecf175fa000p-3, -0x1.4289a7250ee8bp-44, 0.0,
    0x1.b65e2e3beee05p-1, 0x1.cac163c770000p-3, 0x1.b9306bdcc4b5ep-44, 0.0,
    0x1.b37484ad806cep-1, 0x1.de73fe3b14000p-3, 0x1.01b543dfd3c03p-44, 0.0,
    0x1.b094b31d922a4p-1, 0x1.f205339208000p-3, 0x1.e4d4bc06d4602p-44, 0.0,
    0x1.adbe87f94905ep-1, 0x1.02baba24d0000p-2, 0x1.98f0373cd17cbp-44, 0.0,
    0x1.aaf1d2f87ebfdp-1, 0x1.0c62975543000p-2, -0x1.5ca10db5e49e0p-44, 0.0,
    0x1.a82e65130e159p-1, 0x1.15fa676bb1000p-2, -0x1.c07840ed1f4d3p-44, 0.0,
    0x1.a574107688a4ap-1, 0x1.1f825f6d89000p-2, -0x1.ec89126f233adp-46, 0.0,
    0x1.a2c2a87c51ca0p-1, 0x1.28fab35b32000p-2, 0x1.a11e00be8a131p-44, 0.0,
    0x1.a01a01a01a01ap-1, 0x1.32639636b3000p-2, -0x1.f297d5b29971fp-44, 0.0,
    0x1.9d79f176b682dp-1, 0x1.3bbd3a0a1e000p-2, -0x1.824ed00c46a1cp-45, 0.0,
    0x1.9ae24ea5510dap-1, 0x1.4507cfedd5000p-2, -0x1.db3bd7e16ecdcp-49, 0.0,
    0x1.9852f0d8ec0ffp-1, 0x1.4e43880e90000p-2, -0x1.25522d6a89ce3p-44, 0.0,
    0x1.95cbb0be377aep-1, 0x1.577091b338000p-2, -0x1.cdb749e37910ap-44, 0.0,
    0x1.934c67f9b2ce6p-1, 0x1.608f1b4295000p-2, -0x1.d498d2a7ec653p-44, 0.0,
    0x1.90d4f120190d5p-1, 0x1.699f5248cd000p-2, 0x1.2e0c7cafb0fb5p-44, 0.0,
    0x1.8e6527af1373fp-1, 0x1.72a1637cbc000p-2, 0x1.82ae2cc9e6739p-46, 0.0,
    0x1.8bfce8062ff3ap-1, 0x1.7b957ac51b000p-2, -0x1.4ee8b5cf94b1dp-44, 0.0,
    0x1.899c0f601899cp-1, 0x1.847bc33d86000p-2, 0x1.8e0175c76bd1dp-46, 0.0,
    0x1.87427bcc092b9p-1, 0x1.8d54673b5c000p-2, 0x1.b8b46fedf1685p-45, 0.0,
    0x1.84f00c2780614p-1, 0x1.961f905274000p-2, 0x1.35352c5fa9271p-47, 0.0,
    0x1.82a4a0182a4a0p-1, 0x1.9edd6759b2000p-2, 0x1.77f94c0ea39d3p-44, 0.0,
    0x1.8060180601806p-1, 0x1.a78e146f7c000p-2, -0x1.0ba7b8a87d449p-46, 0.0,
    0x1.7e225515a4f1dp-1, 0x1.b031befe06000p-2, 0x1.0d3448a03da91p-44, 0.0,
    0x1.7beb3922e017cp-1, 0x1.b8c88dbf88000p-2, 0x1.9e519ad8dfa81p-44, 0.0,
    0x1.79baa6bb6398bp-1, 0x1.c152a6c24d000p-2, -0x1.46230a2487c7ep-44, 0.0,
    0x1.77908119ac60dp-1, 0x1.c9d02f6ca4000p-2, 0x1.ed2817285162bp-44, 0.0,
    0x1.756cac201756dp-1, 0x1.d2414c80bf000p-2, 0x1.3e0321ee432bfp-45, 0.0,
    0x1.734f0c541fe8dp-1, 0x1.daa6222065000p-2, -0x1.20e56a89ad6dep-48, 0.0,
    0x1.713786d9c7c09p-1, 0x1.e2fed3d097000p-2, 0x1.4b55857dd1de9p-45, 0.0,
    0x1.6f26016f26017p-1, 0x1.eb4b847d16000p-2, -0x1.0c78bb2fea90ep-44, 0.0,
    0x1.6d1a62681c861p-1, 0x1.f38c567bcc000p-2, 0x1.502f32e65692bp-44, 0.0,
    0x1.6b1490aa31a3dp-1, 0x1.fbc16b9027000p-2, -0x1.fd7ab11cc1a4fp-44, 0.0,
    0x1.691473a88d0c0p-1, 0x1.01f5727726800p-1, -0x1.9035112f0c6e4p-44, 0.0,
    0x1.6719f3601671ap-1, 0x1.0604719f25000p-1, -0x1.4ddb5ed132977p-45, 0.0,
    0x1.6524f853b4aa3p-1, 0x1.0a0dc34f8e000p-1, 0x1.fc37cbefc98eap-45, 0.0,
    0x1.63356b88ac0dep-1, 0x1.0e117754d8000p-1, -0x1.f774b755a49adp-44, 0.0,
    0x1.614b36831ae94p-1, 0x1.120f9d39e1800p-1, 0x1.9e997a040d270p-51, 0.0,
    0x1.5f66434292dfcp-1, 0x1.160844495e000p-1, 0x1.72041263716fcp-51, 0.0,
    0x1.5d867c3ece2a5p-1, 0x1.19fb7b8f32800p-1, -0x1.ef0fc3ea8a2f3p-44, 0.0,
    0x1.5babcc647fa91p-1, 0x1.1de951d9cb800p-1, 0x1.d3621447c39d6p-44, 0.0,
    0x1.59d61f123ccaap-1, 0x1.21d1d5bb6d800p-1, -0x1.32ac30fef63b3p-44, 0.0,
    0x1.5805601580560p-1, 0x1.25b5158b74000p-1, -0x1.7dbda7721a483p-44, 0.0,
    0x1.56397ba7c52e2p-1, 0x1.29931f6791800p-1, -0x1.4fecaa06004d0p-44, 0.0,
    0x1.54725e6bb82fep-1, 0x1.2d6c013501000p-1, 0x1.c033c5fb8ab0ep-44, 0.0,
    0x1.52aff56a8054bp-1, 0x1.313fc8a1b3800p-1, -0x1.0e51fec694568p-45, 0.0,
    0x1.50f22e111c4c5p-1, 0x1.350e832570800p-1, -0x1.313528e9e16bbp-48, 0.0,
    0x1.4f38f62dd4c9bp-1, 0x1.38d83e02f6000p-1, -0x1.7bf447bccc154p-44, 0.0,
    0x1.4d843bedc2c4cp-1, 0x1.3c9d06490b000p-1, -0x1.eed558a9cd02dp-45, 0.0,
    0x1.4bd3edda68fe1p-1, 0x1.405ce8d38f800p-1, -0x1.a2290e00170d2p-44, 0.0,
    0x1.4a27fad76014ap-1, 0x1.4417f24c82000p-1, 0x1.6507242272a32p-45, 0.0,
    0x1.4880522014880p-1, 0x1.47ce2f2d02800p-1, -0x1.3c320919f6e22p-44, 0.0,
    0x1.46dce34596066p-1, 0x1.4b7fabbe49800p-1, -0x1.a8bfe9e08f808p-47, 0.0,
    0x1.453d9e2c776cap-1, 0x1.4f2c741a9f000p-1, 0x1.9f3d1993fc134p-44, 0.0,
    0x1.43a2730abee4dp-1, 0x1.52d4942e47800p-1, 0x1.0992c31d3db48p-45, 0.0,
    0x1.420b5265e5951p-1, 0x1.567817b86b000p-1, 0x1.666a9ba8c119ap-48, 0.0,
    0x1.40782d10e6566p-1, 0x1.5a170a4bf9000p-1, -0x1.51e2e6183723ep-44, 0.0,
    0x1.3ee8f42a5af07p-1, 0x1.5db1775084000p-1, 0x1.3bf1c12779b51p-45, 0.0,
    0x1.3d5d991aa75c6p-1, 0x1.61476a031b000p-1, 0x1.07fb1c9997331p-45, 0.0,
    0x1.3bd60d9232955p-1, 0x1.64d8ed7719800p-1, 0x1.f739cefb96710p-44, 0.0,
    0x1.3a524387ac822p-1, 0x1.68660c96f7000p-1, -0x1.df92089b6dd63p-47, 0.0,
    0x1.38d22d366088ep-1, 0x1.6beed2250d000p-1, -0x1.2946b128aefebp-44, 0.0,
    0x1.3755bd1c945eep-1, 0x1.6f7348bc5c800p-1, -0x1.e8ec9fb631d1dp-45, 0.0,
    0x1.35dce5f9f2af8p-1, 0x1.72f37ad14c800p-1, -0x1.27f1cc37d7c43p-44, 0.0,
    0x1.34679ace01346p-1, 0x1.766f72b264000p-1, -0x1.088758521db7ap-44, 0.0,
    0x1.32f5ced6a1dfap-1, 0x1.79e73a8900800p-1, -0x1.e03850c33811dp-45, 0.0,
    0x1.3187758e9ebb6p-1, 0x1.7d5adc5a07800p-1, 0x1.488649c93e7f8p-46, 0.0,
    0x1.301c82ac40260p-1, 0x1.80ca620695000p-1, -0x1.03563758aa866p-44, 0.0,
    0x1.2eb4ea1fed14bp-1, 0x1.8435d54ca3800p-1, -0x1.1825a0a9b3b3bp-46, 0.0,
    0x1.2d50a012d50a0p-1, 0x1.879d3fc7b3800p-1, 0x1.b876474bb5a71p-44, 0.0,
    0x1.2bef98e5a3711p-1, 0x1.8b00aaf16d800p-1, -0x1.ab92e50c4b6c3p-44, 0.0,
    0x1.2a91c92f3c105p-1, 0x1.8e6020223d800p-1, -0x1.9edad4496eb39p-45, 0.0,
    0x1.293725bb804a5p-1, 0x1.91bba891f1800p-1, -0x1.ef469cd65894cp-46, 0.0,
    0x1.27dfa38a1ce4dp-1, 0x1.95134d584e000p-1, 0x1.723ede9377dc6p-44, 0.0,
    0x1.268b37cd60127p-1, 0x1.9867176da3800p-1, 0x1.6b037b598b0e9p-48, 0.0,
    0x1.2539d7e9177b2p-1, 0x1.9bb70fab5d000p-1, -0x1.b333b0e41b705p-45, 0.0,
    0x1.23eb79717605bp-1, 0x1.9f033ecc8e800p-1, 0x1.56e383238f2abp-45, 0.0,
    0x1.22a0122a0122ap-1, 0x1.a24bad6e7f800p-1, 0x1.bb56e4587f881p-44, 0.0,
    0x1.21579804855e6p-1, 0x1.a590641131800p-1, -0x1.4deb9b6c5de8fp-44, 0.0,
    0x1.2012012012012p-1, 0x1.a8d16b17e2800p-1, -0x1.7694c91967ab0p-46, 0.0,
    0x1.1ecf43c7fb84cp-1, 0x1.ac0ecac991000p-1, 0x1.9dd0b679ddfc7p-44, 0.0,
    0x1.1d8f5672e4abdp-1, 0x1.af488b5179000p-1, 0x1.6a34de7dc280cp-44, 0.0,
    0x1.1c522fc1ce059p-1, 0x1.b27eb4bf8f000p-1, 0x1.13c695dca4228p-46, 0.0,
    0x1.1b17c67f2bae3p-1, 0x1.b5b14f08f9800p-1, -0x1.9ae4e4e6cb726p-45, 0.0,
    0x1.19e0119e0119ep-1, 0x1.b8e0620887000p-1, 0x1.84900e72092b4p-44, 0.0,
    0x1.18ab083902bdbp-1, 0x1.bc0bf57f23800p-1, -0x1.fb284658e8807p-45, 0.0,
    0x1.1778a191bd684p-1, 0x1.bf34111446800p-1, -0x1.ac81d319f8fe5p-44, 0.0,
    0x1.1648d50fc3201p-1, 0x1.c258bc5664800p-1, 0x1.4735222ba237cp-48, 0.0,
    0x1.151b9a3fdd5c9p-1, 0x1.c579febb5b800p-1, -0x1.a8bac76a4c10ep-45, 0.0,
    0x1.13f0e8d344724p-1, 0x1.c897dfa0db800p-1, -0x1.3916e3bacd04bp-44, 0.0,
    0x1.12c8b89edc0acp-1, 0x1.cbb2664cd0000p-1, -0x1.85820bb725debp-44, 0.0,
    0x1.11a3019a74826p-1, 0x1.cec999edc5000p-1, 0x1.02249a4cdf070p-44, 0.0,
    0x1.107fbbe011080p-1, 0x1.d1dd819b4c000p-1, 0x1.f8083e73e6927p-44, 0.0,
    0x1.0f5edfab325a2p-1, 0x1.d4ee24565c800p-1, -0x1.d63ca112e4525p-45, 0.0,
    0x1.0e40655826011p-1, 0x1.d7fb8909b2800p-1, 0x1.35fd8cd5c12cep-44, 0.0,
    0x1.0d24456359e3ap-1, 0x1.db05b68a2f800p-1, 0x1.b215d6c600646p-44, 0.0,
    0x1.0c0a7868b4171p-1, 0x1.de0cb39733800p-1, 0x1.465ae94b1a0eep-46, 0.0,
    0x1.0af2f722eecb5p-1, 0x1.e11086daf7800p-1, -0x1.b44e816d6ccddp-44, 0.0,
    0x1.09ddba6af8360p-1, 0x1.e41136eae5800p-1, -0x1.615b783ac1135p-44, 0.0,
    0x1.08cabb37565e2p-1, 0x1.e70eca47ef800p-1, 0x1.bba43a82e5bf1p-47, 0.0,
    0x1.07b9f29b8eae2p-1, 0x1.ea09475ee4000p-1, -0x1.e394d415ed0edp-44, 0.0,
    0x1.06ab59c7912fbp-1, 0x1.ed00b488bf000p-1, -0x1.edcab11a30a2bp-44, 0.0,
    0x1.059eea0727586p-1, 0x1.eff5180afd000p-1, 0x1.f26f189aafaaap-44, 0.0,
    0x1.04949cc1664c5p-1, 0x1.f2e67817eb800p-1, 0x1.1982b58191809p-47, 0.0,
    0x1.038c6b78247fcp-1, 0x1.f5d4dacef3800p-1, -0x1.41cb575dbe016p-45, 0.0,
    0x1.02864fc7729e9p-1, 0x1.f8c0463ce9000p-1, -0x1.cc0bcb9c9ee2ep-44, 0.0,
    0x1.0182436517a37p-1, 0x1.fba8c05c54800p-1, -0x1.8fe922f3df289p-44, 0.0,
    0x1.0000000000000p-1, 0x1.0000000000000p+0, 0x0.0p+0, 0.0,
};
// {2^(j/64), the rest} for j = 0 .. 63
static __device__ const double kPowExp[64 * 2] = {
    0x1.0000000000000p+0, 0x0.0p+0, 0x1.02c9a3e778061p+0, -0x1.19083535b085dp-56,
    0x1.059b0d3158574p+0, 0x1.d73e2a475b465p-55, 0x1.0874518759bc8p+0, 0x1.186be4bb284ffp-57,
    0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54, 0x1.0e3ec32d3d1a2p+0, 0x1.03a1727c57b53p-59,
    0x1.11301d0125b51p+0, -0x1.6c51039449b3ap-54, 0x1.1429aaea92de0p+0, -0x1.32fbf9af1369ep-54,
    0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55, 0x1.1a35beb6fcb75p+0, 0x1.e5b4c7b4968e4p-55,
    0x1.1d4873168b9aap+0, 0x1.e016e00a2643cp-54, 0x1.2063b88628cd6p+0, 0x1.dc775814a8495p-55,
    0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54, 0x1.26b4565e27cddp+0, 0x1.2bd339940e9d9p-55,
    0x1.29e9df51fdee1p+0, 0x1.612e8afad1255p-55, 0x1.2d285a6e4030bp+0, 0x1.0024754db41d5p-54,
    0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55, 0x1.33c08b26416ffp+0, 0x1.32721843659a6p-54,
    0x1.371a7373aa9cbp+0, -0x1.63aeabf42eae2p-54, 0x1.3a7db34e59ff7p+0, -0x1.5e436d661f5e3p-56,
    0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55, 0x1.4160a21f72e2ap+0, -0x1.ef3691c309278p-58,
    0x1.44e086061892dp+0, 0x1.89b7a04ef80d0p-59, 0x1.486a2b5c13cd0p+0, 0x1.3c1a3b69062f0p-56,
    0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56, 0x1.4f9b2769d2ca7p+0, -0x1.4b309d25957e3p-54,
    0x1.5342b569d4f82p+0, -0x1.07abe1db13cadp-55, 0x1.56f4736b527dap+0, 0x1.9bb2c011d93adp-54,
    0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54, 0x1.5e76f15ad2148p+0, 0x1.ba6f93080e65ep-54,
    0x1.6247eb03a5585p+0, -0x1.383c17e40b497p-54, 0x1.6623882552225p+0, -0x1.bb60987591c34p-54,
    0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54, 0x1.6dfb23c651a2fp+0, -0x1.bbe3a683c88abp-57,
    0x1.71f75e8ec5f74p+0, -0x1.16e4786887a99p-55, 0x1.75feb564267c9p+0, -0x1.0245957316dd3p-54,
    0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55, 0x1.7e2f336cf4e62p+0, 0x1.05d02ba15797ep-56,
    0x1.82589994cce13p+0, -0x1.d4c1dd41532d8p-54, 0x1.868d99b4492edp+0, -0x1.fc6f89bd4f6bap-54,
    0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54, 0x1.8f1ae99157736p+0, 0x1.5cc13a2e3976cp-55,
    0x1.93737b0cdc5e5p+0, -0x1.75fc781b57ebcp-57, 0x1.97d829fde4e50p+0, -0x1.d185b7c1b85d1p-54,
    0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56, 0x1.a0c667b5de565p+0, -0x1.359495d1cd533p-54,
    0x1.a5503b23e255dp+0, -0x1.d2f6edb8d41e1p-54, 0x1.a9e6b5579fdbfp+0, 0x1.0fac90ef7fd31p-54,
    0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54, 0x1.b33a2b84f15fbp+0, -0x1.2805e3084d708p-57,
    0x1.b7f76f2fb5e47p+0, -0x1.5584f7e54ac3bp-56, 0x1.bcc1e904bc1d2p+0, 0x1.23dd07a2d9e84p-55,
    0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55, 0x1.c67f12e57d14bp+0, 0x1.2884dff483cadp-54,
    0x1.cb720dcef9069p+0, 0x1.503cbd1e949dbp-56, 0x1.d072d4a07897cp+0, -0x1.cbc3743797a9cp-54,
    0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55, 0x1.da9e603db3285p+0, 0x1.c2300696db532p-54,
    0x1.dfc97337b9b5fp+0, -0x1.1a5cd4f184b5cp-54, 0x1.e502ee78b3ff6p+0, 0x1.39e8980a9cc8fp-55,
    0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54, 0x1.efa1bee615a27p+0, 0x1.dc7f486a4b6b0p-54,
    0x1.f50765b6e4540p+0, 0x1.9d3e12dd8a18bp-54, 0x1.fa7c1819e90d8p+0, 0x1.74853f3a5931ep-55,
};

// the tables in LDS, one copy per block
struct PowTab {
  double lg[128 * 4];
  double ex[64 * 2];
};

__device__ __forceinline__ void load_pow_tab(PowTab &t) {
  for (int k = threadIdx.x; k < 128 * 4; k += blockDim.x) t.lg[k] = kPowLog[k];
  for (int k = threadIdx.x; k < 64 * 2; k += blockDim.x) t.ex[k] = kPowExp[k];
  __syncthreads();
}

__device__ __forceinline__ double pow_tab(const PowTab &t, double x, double y) {
  const long long bits = __double_as_longlong(x);
  const int hiw = (int)(bits >> 32);
  const int e = (hiw >> 20) - 1023;
  const int i = (hiw >> 13) & 127;
  const double m = __hiloint2double((hiw & 0xfffff) | 0x3ff00000, (int)bits);
  const double *L = t.lg + 4 * i;
  const double r = fma(m, L[0], -1.0);
  // log2(1 + r) = r / ln 2 (two doubles) + r^2 q(r)
  const double kInvLn2 = 0x1.71547652b82fep+0, kInvLn2Lo = 0x1.777d0ffda0d24p-56;
  const double u = r * kInvLn2;
  const double ul = fma(r, kInvLn2Lo, fma(r, kInvLn2, -u));
  const double r2 = r * r;
  const double q0 = fma(r, 0x1.ec709dc3a03fdp-2, -0x1.71547652b82fep-1);
  const double q1 = fma(r, 0x1.2776c50ef9bfep-2, -0x1.71547652b82fep-2);
  const double q2 = fma(r, 0x1.a61762a7aded9p-3, -0x1.ec709dc3a03fdp-3);
  const double q = fma(r2, fma(r2, fma(r2, -0x1.71547652b82fep-3, q2), q1), q0);
  const double h = (double)e + L[1];
  const double s = h + u;
  const double lo = ((u - (s - h)) + (ul + L[2])) + r2 * q;
  const double z = y * s;
  const double zl = fma(y, lo, fma(y, s, -z));
  const double kd = rint(z * 64.0);
  const int k = (int)kd;
  const double f = fma(kd, -0.015625, z) + zl;
  const double *E2 = t.ex + 2 * (k & 63);
  const double f2 = f * f;
  const double p0 = fma(f, 0x1.ebfbdff82c58fp-3, 0x1.62e42fefa39efp-1);
  const double p1 = fma(f, 0x1.3b2ab6fba4e77p-7, 0x1.c6b08d704a0c0p-5);
  const double p2 = fma(f, 0x1.430912f86c787p-13, 0x1.5d87fe78a6731p-10);
  const double p = f * fma(f2, fma(f2, p2, p1), p0);
  return ldexp(E2[0] + fma(E2[0], p, E2[1]), k >> 6);
}

// pow_abs of sq_device.h for x = |x|: 1 for a zero exponent or base 1, 0 for
// base 0 (to 1e-12); a base that has left every scale stays out of range
__device__ __forceinline__ double q_pow(const PowTab &t, double x, double y) {
  const double tol = 1e-12;
  double r = pow_tab(t, x, y);
  r = x < 1e300 ? r : (y > 0.0 ? x * x : 1.0 / (x * x));
  r = x < tol ? 0.0 : r;
  r = (fabs(y) < tol || fabs(x - 1.0) < tol) ? 1.0 : r;
  return r;
}

}  // namespace sqd
