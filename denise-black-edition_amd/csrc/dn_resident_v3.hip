// Chip-resident time loop, FDORDER 6, viscoelastic P/SV.
#define DN_F 3
#define DN_GROUP 2
#include "dn_resident_inst.inc"
