// The x line's plans (variants 4 and 5), replayed as fft2_emul.cpp replays the rest.
#define main fft2_emul_main
#include "fft2_emul.cpp"
#undef main

int main() {
  RUNV(16, 4) RUNV(24, 4) RUNV(32, 4) RUNV(96, 4) RUNV(16, 5) RUNV(24, 5) RUNV(32, 5) RUNV(96, 5)
  return 0;
}
