// The checks of test_lds_layout.cpp for the k-major layouts whose 16-byte instruction spans
// several k-rows (FP32 up to 128 rows, FP64 64 rows) and for the 256-row FP32 tile.
#define main lds_layout_main
#include "test_lds_layout.cpp"
#undef main

int main() {
    static_assert(SlabLayout<float, 128, 16, false, true>::KPI == 2 && SlabLayout<float, 64, 16, false, true>::KPI == 4 &&
                  SlabLayout<double, 64, 16, false, true>::KPI == 2 && SlabLayout<double, 128, 16, false, true>::KPI == 1);
    static_assert(kmajor_wide<float>(64) && kmajor_wide<float>(128) && kmajor_wide<float>(256) && kmajor_wide<double>(64) &&
                  kmajor_wide<double>(128) && !kmajor_wide<double>(96) && !kmajor_wide<float>(96));
    check_layout<double, 64, 16, false, true>("f64 64 kmajor x4");
    check_layout<float, 64, 16, false, true>("f32 64 kmajor x4");
    check_layout<float, 128, 16, false, true>("f32 128 kmajor x4");
    check_layout<float, 256, 16, false, false>("f32 256 kmajor dword");
    check_layout<float, 256, 16, false, true>("f32 256 kmajor x4");
    check_layout<float, 256, 16, true, false>("f32 256 krow dword");
    check_layout<float, 256, 16, true, true>("f32 256 krow x4");
    std::printf("%d failures\n", failures);
    return failures ? 1 : 0;
}
