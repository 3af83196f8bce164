// Generated by gen_constants.py -- do not edit.
#pragma once
#include <stdint.h>
namespace fk20 {

// ---- Fp: 14 x 29-bit limbs, Montgomery radix 2^406 ----
static constexpr int FP_N = 14;
static constexpr uint32_t FP_MASK = 0x1fffffffu;
static constexpr uint32_t FP_P[14] = {0x1fffaaabu, 0x0ff7ffffu, 0x14ffffeeu, 0x17fffd62u, 0x0f6241eau, 0x09507b58u, 0x0afd9cc3u, 0x109e70a2u, 0x1764774bu, 0x121a5d66u, 0x12c6e9edu, 0x12ffcd34u, 0x00111ea3u, 0x0000000du};
static constexpr uint32_t FP_PINV = 0x1ffcfffdu;  // -p^-1 mod 2^29
static constexpr uint32_t FP_R2[14] = {0x15bef7aeu, 0x1031cd0eu, 0x02dd93e8u, 0x09226323u, 0x0e6e2cd2u, 0x11684daau, 0x1170e5dbu, 0x088e25b1u, 0x1b366399u, 0x1c536f47u, 0x0d1f9cbcu, 0x0278b67fu, 0x1ea66a2bu, 0x0000000cu};  // R^2 mod p
static constexpr uint32_t FP_ONE[14] = {0x03a9fb84u, 0x0ba00690u, 0x071288f1u, 0x0f59bcc5u, 0x126cb614u, 0x0585bf36u, 0x1b85ac3du, 0x1cf856fau, 0x1891ecbdu, 0x1a7eec05u, 0x155a88f0u, 0x0741ac6du, 0x1317c30fu, 0x00000009u};  // R mod p
static constexpr uint32_t FP_2P[14] = {0x1fff5556u, 0x1fefffffu, 0x09ffffdcu, 0x0ffffac5u, 0x1ec483d5u, 0x12a0f6b0u, 0x15fb3986u, 0x013ce144u, 0x0ec8ee97u, 0x0434bacdu, 0x058dd3dbu, 0x05ff9a69u, 0x00223d47u, 0x0000001au};  // 2 p
static constexpr uint32_t FP_4P[14] = {0x1ffeaaacu, 0x1fdfffffu, 0x13ffffb9u, 0x1ffff58au, 0x1d8907aau, 0x0541ed61u, 0x0bf6730du, 0x0279c289u, 0x1d91dd2eu, 0x0869759au, 0x0b1ba7b6u, 0x0bff34d2u, 0x00447a8eu, 0x00000034u};  // 4 p
static constexpr uint32_t FP_8P[14] = {0x1ffd5558u, 0x1fbfffffu, 0x07ffff73u, 0x1fffeb15u, 0x1b120f55u, 0x0a83dac3u, 0x17ece61au, 0x04f38512u, 0x1b23ba5cu, 0x10d2eb35u, 0x16374f6cu, 0x17fe69a4u, 0x0088f51cu, 0x00000068u};  // 8 p
static constexpr uint32_t FP_16P[14] = {0x1ffaaab0u, 0x1f7fffffu, 0x0ffffee7u, 0x1fffd62au, 0x16241eabu, 0x1507b587u, 0x0fd9cc34u, 0x09e70a25u, 0x164774b8u, 0x01a5d66bu, 0x0c6e9ed9u, 0x0ffcd349u, 0x0111ea39u, 0x000000d0u};  // 16 p
static constexpr uint32_t FP_32P[14] = {0x1ff55560u, 0x1effffffu, 0x1ffffdcfu, 0x1fffac54u, 0x0c483d57u, 0x0a0f6b0fu, 0x1fb39869u, 0x13ce144au, 0x0c8ee970u, 0x034bacd7u, 0x18dd3db2u, 0x1ff9a692u, 0x0223d472u, 0x000001a0u};  // 32 p
static constexpr uint32_t FP_64P[14] = {0x1feaaac0u, 0x1dffffffu, 0x1ffffb9fu, 0x1fff58a9u, 0x18907aafu, 0x141ed61eu, 0x1f6730d2u, 0x079c2895u, 0x191dd2e1u, 0x069759aeu, 0x11ba7b64u, 0x1ff34d25u, 0x0447a8e5u, 0x00000340u};  // 64 p
static constexpr uint32_t FP_128P[14] = {0x1fd55580u, 0x1bffffffu, 0x1ffff73fu, 0x1ffeb153u, 0x1120f55fu, 0x083dac3du, 0x1ece61a5u, 0x0f38512bu, 0x123ba5c2u, 0x0d2eb35du, 0x0374f6c8u, 0x1fe69a4bu, 0x088f51cbu, 0x00000680u};  // 128 p
static constexpr uint64_t GLV_LAMBDA[2] = {0x00000000ffffffffull, 0xac45a4010001a402ull};  // z^2 - 1

// ---- Fp, signed form: 13 x 30-bit digits, Montgomery radix 2^390 ----
static constexpr int FQ_N = 13;
static constexpr uint32_t FQ_MASK = 0x3fffffffu;
static constexpr int32_t FQ_P[13] = {-21845, -402915328, 356515836, -352321620, -252304353, 55215067, 288093811, 316751073, -321428361, 517541167, -375082566, -91332614, 1704210};  // p
static constexpr int32_t FQ_PT[14] = {-1, 135004164, 5054525, -327173, 12685220, -359651098, -383584983, 280525645, 202633227, -68632997, -303925084, -261624741, -58966498, -312};  // -196611 p: digit 0 is -1
// (-p^-1 mod 2^30) << 2: a low word times this, shifted right by 2, is the signed quotient digit
static constexpr uint32_t FQ_PINV4 = 0xfff3fff4u;
static constexpr int64_t FQ_K0 = 6969937068335403541ll;
static constexpr int32_t FQ_BETA[13] = {550457077, 529115271, 538425416, 540408362, 534947505, 530527195, 527739787, 553457329, 541486612, 537384151, 545225655, 547666669, 37975};  // digit offsets of a product
static constexpr int32_t FQ_ONE[13] = {13762350, 433586176, -192935228, -301937177, 37952645, -425753694, -36732706, 162803105, -437337492, 366579475, 78814996, -442511456, 89578};  // R mod p
static constexpr int32_t FQ_R2[13] = {84958308, 320669453, -336452545, -23350980, 68258640, -130586467, 277172093, -144228653, 171105485, -419190883, -282802362, -41659541, -694179};  // R^2 mod p
static constexpr int32_t FQ_R3[13] = {323471757, -333343540, 453147883, -343099995, 303348703, 190774532, -101855041, 455817637, -223343770, 488336821, -74511473, 315118520, 446639};  // R^3 mod p
static constexpr int32_t FQ_GLV[13] = {479228289, -54664058, -430486465, -215714323, 473873436, -101816220, 385853527, -332097025, 89177367, 348892208, 399608966, -514237961, 640725};  // beta of the endomorphism (Montgomery)
static constexpr int32_t FQ_GLV2[13] = {-492990639, -378922118, -450320131, 517651501, -511826081, 527569914, -349120821, 169293920, 348160125, 358270141, -478423963, -116992407, -730302};  // beta^2
static constexpr int32_t FQ_4P[13] = {1073654444, 535822335, 352321518, 738197169, 64524410, 220860267, 78633420, 193262469, 861770205, 996422842, 647153385, 708411366, 6816839};  // 4 p, non-negative digits
static constexpr uint32_t FQ_FROM_FP[14] = {0x00d1ff2eu, 0x13b00000u, 0x12002b11u, 0x10066f36u, 0x0431c84bu, 0x13f07441u, 0x13e03766u, 0x1a16d07bu, 0x0ec26c26u, 0x131e252fu, 0x0a7c515du, 0x1e7d0096u, 0x15de9967u, 0x00000000u};  // 2^390 mod p: x 2^406 -> x 2^390
static constexpr uint32_t FP_FROM_FQ[14] = {0x1a7f6bafu, 0x1e281d51u, 0x19fe47cbu, 0x16b3408eu, 0x136783f9u, 0x0d3c8407u, 0x1e61f415u, 0x15deb981u, 0x10c53570u, 0x0067aa9du, 0x0256511cu, 0x08eb4399u, 0x004f0125u, 0x00000002u};  // 2^422 mod p: x 2^390 -> x 2^406

// p as 12 x 32-bit limbs (packed storage form)
static constexpr uint32_t FP_P_PACKED[12] = {0xffffaaabu, 0xb9feffffu, 0xb153ffffu, 0x1eabfffeu, 0xf6b0f624u, 0x6730d2a0u, 0xf38512bfu, 0x64774b84u, 0x434bacd7u, 0x4b1ba7b6u, 0x397fe69au, 0x1a0111eau};
static constexpr uint32_t FP_HALF_PACKED[12] = {0xffffd555u, 0xdcff7fffu, 0x58a9ffffu, 0x0f55ffffu, 0x7b587b12u, 0xb3986950u, 0x79c2895fu, 0xb23ba5c2u, 0x21a5d66bu, 0x258dd3dbu, 0x1cbff34du, 0x0d0088f5u};  // (p - 1) / 2: y above it is the larger root
// the 12 x 32-bit CIOS layout of the limb-layout probe (Montgomery radix 2^384)
static constexpr const uint32_t *FP32_P = FP_P_PACKED;
static constexpr uint32_t FP32_PINV = 0xfffcfffdu;  // -p^-1 mod 2^32

// ---- Fr: 8 x 32-bit limbs, Montgomery radix 2^256 ----
static constexpr uint32_t FR_R[8] = {0x00000001u, 0xffffffffu, 0xfffe5bfeu, 0x53bda402u, 0x09a1d805u, 0x3339d808u, 0x299d7d48u, 0x73eda753u};
static constexpr uint32_t FR_RINV = 0xffffffffu;  // -r^-1 mod 2^32
static constexpr uint32_t FR_R2[8] = {0xf3f29c6du, 0xc999e990u, 0x87925c23u, 0x2b6cedcbu, 0x7254398fu, 0x05d31496u, 0x9f59ff11u, 0x0748d9d9u};  // 2^512 mod r
static constexpr uint32_t FR_ONE[8] = {0xfffffffeu, 0x00000001u, 0x00034802u, 0x5884b7fau, 0xecbc4ff5u, 0x998c4fefu, 0xacc5056fu, 0x1824b159u};  // 2^256 mod r
static constexpr uint32_t FR_RM2[8] = {0xffffffffu, 0xfffffffeu, 0xfffe5bfeu, 0x53bda402u, 0x09a1d805u, 0x3339d808u, 0x299d7d48u, 0x73eda753u};  // r - 2 (Fermat inverse exponent)
// Fr of the transforms: 9 x 29-bit digits, Montgomery radix 2^261
static constexpr int32_t FN_RT[9] = {-1, 8, 6881344, 79165952, 41921220, -201589969, 182399769, -174404528, -7597479};  // -r: digit 0 is -1
static constexpr uint32_t FP_PM2[12] = {0xffffaaa9u, 0xb9feffffu, 0xb153ffffu, 0x1eabfffeu, 0xf6b0f624u, 0x6730d2a0u, 0xf38512bfu, 0x64774b84u, 0x434bacd7u, 0x4b1ba7b6u, 0x397fe69au, 0x1a0111eau};  // p - 2 (Fermat inverse exponent)

}  // namespace fk20
